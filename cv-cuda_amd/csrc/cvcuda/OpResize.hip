// Resize with nearest / bilinear / bicubic / area sampling, tensors and var-shape batches.
//
// Index maps and weights follow the reference kernels expression for expression in float32
// (src/cvcuda/priv/OpResize.cu:142-164 nearest, 177-330 bilinear, 334-388 bicubic;
// src/cvcuda/priv/legacy/resize_var_shape.cu:92-231 for the var-shape association of the sums).
// The nearest-neighbour source index uses the single-multiply form floor((d+.5f)*scale) of the
// reference's CPU golden (tests/cvcuda/system/ResizeUtils.cpp:206-221) for every pixel, so results
// are bit-exact against it also where the coordinate lands on an integer. 8-bit pixels are blended in fixed
// point on those indices and weights (bilinear: FixedPointBlend.hpp; bicubic: kFixedCubic; box filter:
// kAreaFixed), at most 1 from the reference's goldens.
//
// Ten kernel shapes, all with streaming stores, var-shape batches on a packed tile grid:
//  * pixels of up to 8 bytes: wave patches (64 columns x 4 rows per wave; adjacent taps in one load,
//    row terms computed once per wave, 4x4 lane transposes so that every lane stores whole dwords);
//  * 8-bit bilinear at horizontal scales up to 2: a lane owns 2 columns x 4 rows (image batches x 2; 4 x 8 when
//    enlarging by 1.5 or more) and fetches each source row once for all its columns and rows, lane pairs swap a
//    pixel pair each;
//    nearest neighbour takes the same strips when enlarging by 1.5 or more;
//  * 8-bit bicubic at vertical scales up to 4, launches of 1024 waves and more (image batches: 3 and 4 channels, 2048
//    blocks): a wave walks down the source rows once, keeps the sums of the last four and finishes output rows as it goes;
//  * bicubic reductions >= 2x of 12/16-byte pixels: tap-major loads exchanged through LDS;
//  * AREA of 8-bit pixels at reductions of up to 3: fixed-point row sums, a wave owns 64 columns x 16 rows and
//    produces vertically adjacent rows in pairs from the source rows they share;
//  * AREA of 8-bit tensors at larger reductions: one lane per output pixel, a row of its box in one window, rows in
//    batches;
//  * bilinear one-channel float tensors whose rows are not reduced, launches of 704 blocks and more: whole rows
//    gathered in LDS and written out on 64-byte boundaries;
//  * AREA of float tensors at reductions: a wave sums the rows of 64 boxes column by column, then each lane its box's
//    columns (ResizeAreaFloatKernel);
//  * bicubic float tensors at scales below 2, large launches: a wave owns 64 columns x 16 rows and forms every source
//    row's sums once (ResizeCubicStripF32Kernel);
//  * everything else (other 12/16-byte pixels, other AREA): one lane per output pixel, a 256-thread block covers
//    64 columns x 4 rows, pixels moved as whole C-channel vectors.
#include "DeviceUtils.hpp"
#include "FixedPointBlend.hpp"
#include "LaneExchange.hpp"
#include "LinearRows.hpp"
#include "OpCommon.hpp"
#include "RunIO.hpp"
#include "VarShapeTiles.hpp"
#include "WaveOrder.hpp"

#include <cvcuda/OpResize.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace cvamd {

namespace {

constexpr int kTileW = 64;
constexpr int kTileH = 4;

template<class T, int C>
using Pixel = Packed<T, C>;

struct ResizeArgs
{
    // tensors
    const uint8_t *srcBase;
    uint8_t       *dstBase;
    int64_t        srcSampleStride, dstSampleStride;
    int32_t        srcRowStride, dstRowStride;
    int32_t        srcW, srcH, dstW, dstH;
    float          scaleX, scaleY; // srcW / dstW, srcH / dstH in float32 (var-shape: per image, in the kernel)
    // var-shape
    const NVCVImageBufferStrided *srcList;
    const NVCVImageBufferStrided *dstList;
};

struct Plane
{
    const uint8_t *src;
    uint8_t       *dst;
    int32_t        srcRow, dstRow, srcW, srcH, dstW, dstH;
    float          scaleX, scaleY;
};

template<bool VARSHAPE>
__device__ __forceinline__ Plane GetPlanes(const ResizeArgs &a, int n)
{
    Plane p;
    if constexpr (VARSHAPE)
    {
        const NVCVImagePlaneStrided &s = a.srcList[n].planes[0];
        const NVCVImagePlaneStrided &d = a.dstList[n].planes[0];
        p = {AsGlobal(s.basePtr),
             AsGlobal(d.basePtr),
             s.rowStride,
             d.rowStride,
             s.width,
             s.height,
             d.width,
             d.height,
             static_cast<float>(s.width) / d.width,
             static_cast<float>(s.height) / d.height};
    }
    else
    {
        p = {a.srcBase + n * a.srcSampleStride,
             a.dstBase + n * a.dstSampleStride,
             a.srcRowStride,
             a.dstRowStride,
             a.srcW,
             a.srcH,
             a.dstW,
             a.dstH,
             a.scaleX,
             a.scaleY};
    }
    return p;
}

template<class T, int C>
__device__ __forceinline__ Pixel<T, C> LoadPx(const uint8_t *row, int x)
{
    return reinterpret_cast<const Pixel<T, C> *>(row)[x];
}

template<class T, int C>
__device__ __forceinline__ void StorePx(uint8_t *row, int x, const Pixel<T, C> &px)
{
    Pixel<T, C> *p = reinterpret_cast<Pixel<T, C> *>(row) + x;
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        __builtin_nontemporal_store(px.v[c], &p->v[c]);
    }
}

// N horizontally adjacent pixels at byte offset `xoff` of source row `row` (all inside the image).
// u8x3: 1 or 2 pixels are fetched with a 4- or 8-byte load that reads 1-2 bytes past them, harmless
// except behind the image's last row (`lastRow`, wave-uniform), where the load is moved back to end
// with the row's `rowBytes` and the value shifted; rows shorter than the load are read byte by byte.
template<class T, int C, int N>
__device__ __forceinline__ void LoadTaps(const uint8_t *row, int xoff, bool lastRow, int rowBytes, float (&t)[N][C])
{
    if constexpr (std::is_same_v<T, uint8_t> && C == 3 && N == 1)
    {
        uint32_t q;
        if (lastRow && rowBytes < 4) // a 1-pixel-wide image: moving the load back would leave the row (and a 1 x 1 image)
        {
            q = row[xoff] | (row[xoff + 1] << 8) | (row[xoff + 2] << 16);
        }
        else if (lastRow)
        {
            const int back = max(0, xoff - (rowBytes - 4));
            q              = LoadU32Unaligned(row + (xoff - back)) >> (8 * back);
        }
        else
        {
            q = LoadU32Unaligned(row + xoff);
        }
        t[0][0] = (float)(q & 0xFF);
        t[0][1] = (float)((q >> 8) & 0xFF);
        t[0][2] = (float)((q >> 16) & 0xFF);
    }
    else if constexpr (std::is_same_v<T, uint8_t> && C == 3 && N == 2)
    {
        uint64_t q;
        if (lastRow && rowBytes < 8) // a 2-pixel-wide image (the two taps are all of the row)
        {
            q = 0;
#pragma unroll
            for (int i = 0; i < 6; ++i)
            {
                q |= (uint64_t)row[xoff + i] << (8 * i);
            }
        }
        else if (lastRow)
        {
            const int back = max(0, xoff - (rowBytes - 8));
            q              = LoadU64Unaligned(row + (xoff - back)) >> (8 * back);
        }
        else
        {
            q = LoadU64Unaligned(row + xoff);
        }
        const uint32_t lo = (uint32_t)q, hi = (uint32_t)(q >> 32);
        t[0][0] = (float)(lo & 0xFF);
        t[0][1] = (float)((lo >> 8) & 0xFF);
        t[0][2] = (float)((lo >> 16) & 0xFF);
        t[1][0] = (float)(lo >> 24);
        t[1][1] = (float)(hi & 0xFF);
        t[1][2] = (float)((hi >> 8) & 0xFF);
    }
    else
    {
        const Pixel<T, N *C> v = *reinterpret_cast<const Pixel<T, N * C> *>(row + xoff);
#pragma unroll
        for (int i = 0; i < N; ++i)
        {
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                t[i][c] = (float)v.v[i * C + c];
            }
        }
    }
}

// Two horizontally adjacent 8-bit pixels as raw bytes (byte i of {w[1]:w[0]} = channel i % C of pixel i / C);
// the same loads as LoadTaps<uint8_t, C, 2>.
template<int C>
__device__ __forceinline__ void LoadTapPairBytes(const uint8_t *row, int xoff, bool lastRow, int rowBytes, uint32_t (&w)[2])
{
    if constexpr (C == 3)
    {
        uint64_t q;
        if (lastRow && rowBytes < 8)
        {
            q = 0;
#pragma unroll
            for (int i = 0; i < 6; ++i)
            {
                q |= (uint64_t)row[xoff + i] << (8 * i);
            }
        }
        else if (lastRow)
        {
            const int back = max(0, xoff - (rowBytes - 8));
            q              = LoadU64Unaligned(row + (xoff - back)) >> (8 * back);
        }
        else
        {
            q = LoadU64Unaligned(row + xoff);
        }
        w[0] = (uint32_t)q;
        w[1] = (uint32_t)(q >> 32);
    }
    else
    {
        const Pixel<uint8_t, 2 * C> v = *reinterpret_cast<const Pixel<uint8_t, 2 * C> *>(row + xoff);
        w[0] = w[1] = 0;
        __builtin_memcpy(w, &v, 2 * C);
    }
}

// Bytes from the dword boundary in front of a row to the row (wave-uniform).
__device__ __forceinline__ uint32_t RowMisalignment(const uint8_t *row)
{
    return (uint32_t)reinterpret_cast<uintptr_t>(row) & 3u;
}

// Four horizontally adjacent 8-bit pixels as raw bytes (the box filter's and the bicubic blend's row window): the
// D dwords that hold the 4 pixels at byte offset `at` + `shift` of the row (`at` a multiple of 4, shift 0 .. 3; 4 channels:
// any, none), brought to the front: pixel k, channel c in byte k * C + c.
// ODD: rows may start at other places than dwords of memory. Loads counted from an odd row are not dword aligned, and the
// vector memory path takes those apart (32 x 1921 x 1081 -> 1280 x 720, box filter: 137 us counted from the row, 78 us from the
// dword of memory); finding that dword costs two vector and a few scalar instructions per row, which images whose rows are
// aligned do without (64 x 256 x 256 u8x3 -> 224 x 224 bicubic 15.9 us with them, 14.0 without; 16 x 720p -> 1080p u8x1 50.3
// and 46.9). The launch chooses (RowsAreOdd): one kernel that holds both forms takes the registers of the larger (16 x 1080p
// -> 1000 x 500 u8x1, box filter: 22.4 us, 31.3 in one kernel).
template<int C, bool GUARDED, bool ODD>
__device__ __forceinline__ void LoadQuadWindow(const uint8_t *row, uint32_t at, uint32_t shift, bool lastRow, uint32_t rowBytes,
                                               uint32_t (&r)[C])
{
    constexpr int D = C == 4 ? 4 : C + 1;
    struct __attribute__((packed, aligned(1))) Window
    {
        uint32_t d[D];
    };
    if constexpr (C == 4)
    {
        const Window w = *reinterpret_cast<const Window *>(row + at);
        __builtin_memcpy(r, &w, 16);
    }
    else
    {
        // the load runs up to 4 bytes past the window, harmless except behind the image's last row, where it is counted
        // from the row and moved back to end with it (GUARDED: the rows passed may include that one)
        // (wave-uniform, but without a branch: with one the compiler kept the places of all of a pixel's rows, 117 registers
        // for 61)
        const bool     guard = GUARDED && lastRow;
        const uint32_t mis   = ODD && !guard ? RowMisalignment(row) : 0u, o = at + shift + mis;
        uint32_t       from  = ODD ? o & ~3u : at;
        from                 = guard ? min(from, rowBytes - 4 * D) : from;
        const Window   w     = *reinterpret_cast<const Window *>(row - mis + from);
        const uint32_t sh    = GUARDED ? o - from : ODD ? o : shift; // (its low two bits count; 4 only if moved back)
        const bool     whole = GUARDED && sh == 4;
#pragma unroll
        for (int i = 0; i < C; ++i)
        {
            r[i] = __builtin_amdgcn_alignbyte(w.d[i + 1], w.d[i], sh);
            if constexpr (GUARDED)
            {
                r[i] = whole ? w.d[i + 1] : r[i];
            }
        }
    }
}

// Channel c of pixels ka and ka + 1 of such a window as (first | second << 16).
template<int C>
__device__ __forceinline__ uint32_t QuadTapPair(const uint32_t (&r)[C], int ka, int c)
{
    const int      b0 = ka * C + c, b1 = b0 + C, j = b0 / 4;
    const uint32_t sel = 0x0c000c00u | (uint32_t)(b0 - 4 * j) | ((uint32_t)(b1 - 4 * j) << 16);
    return __builtin_amdgcn_perm(r[j + 1 < C ? j + 1 : C - 1], r[j], sel);
}

__device__ __forceinline__ void CubicCoeffs(float d, float (&w)[4])
{
    constexpr float A = -0.75f;
    w[0]              = ((A * (d + 1) - 5 * A) * (d + 1) + 8 * A) * (d + 1) - 4 * A;
    w[1]              = ((A + 2) * d - (A + 3)) * d * d + 1;
    w[2]              = ((A + 2) * (1 - d) - (A + 3)) * (1 - d) * (1 - d) + 1;
    w[3]              = 1.f - w[0] - w[1] - w[2];
}

// 8-bit pixels are blended bilinearly in 15-bit fixed point (FixedPointBlend.hpp), tensors and image
// batches alike, whichever kernel form a shape takes: the weight of the second tap along an axis (0 .. 1,
// the reference's float32 expression) is cut to a multiple of 2^-15.
template<class T>
constexpr bool kFixedLinear = std::is_same_v<T, uint8_t>;

// 8-bit pixels are blended bicubically with the four horizontal weights (the reference's float32 polynomials)
// rounded to multiples of 2^-14, the last one taking the remainder so that they add up to exactly 1; a row's four
// taps are combined in integers (exact), the four row sums in float32 with the vertical weights, ascending, by
// fused multiply-adds; the magnitude is rounded once. Tensors and image batches alike, whichever kernel form a
// shape takes. Within 0.05 of the float32 expression, i.e. at most 1 from the reference's golden.
template<class T>
constexpr bool kFixedCubic = std::is_same_v<T, uint8_t>;

__device__ __forceinline__ uint32_t FractionQ15(float w)
{
    return (uint32_t)(w * 32768.f);
}

template<class T, int C, int INTERP, bool VARSHAPE>
__device__ __forceinline__ Pixel<T, C> ResizeValue(const Plane &p, int dx, int dy)
{
    const float scaleX = p.scaleX, scaleY = p.scaleY;
    Pixel<T, C> out;

    if constexpr (INTERP == NVCV_INTERP_NEAREST)
    {
        const int sx = min((int)floorf(scaleX * (dx + 0.5f)), p.srcW - 1);
        const int sy = min((int)floorf(scaleY * (dy + 0.5f)), p.srcH - 1);
        out          = LoadPx<T, C>(p.src + (int64_t)sy * p.srcRow, sx);
    }
    else if constexpr (INTERP == NVCV_INTERP_LINEAR)
    {
        const float fx = (dx + .5f) * scaleX - .5f;
        const float fy = (dy + .5f) * scaleY - .5f;
        int         sx = (int)floorf(fx);
        int         sy = (int)floorf(fy);
        const float wx = (sx < 0) ? 0.f : ((sx > p.srcW - 2) ? 1.f : fx - sx);
        const float wy = (sy < 0) ? 0.f : ((sy > p.srcH - 2) ? 1.f : fy - sy);
        sx             = max(0, min(sx, p.srcW - 2));
        sy             = max(0, min(sy, p.srcH - 2));
        // a 1-pixel-wide (or -high) source has no second tap: reuse the first (its weight is then 0 or
        // multiplies an equal value)
        const int sx1 = min(sx + 1, p.srcW - 1);
        sx            = max(sx, 0);
        const uint8_t *r0 = p.src + (int64_t)max(sy, 0) * p.srcRow;
        const uint8_t *r1 = p.src + (int64_t)min(sy + 1, p.srcH - 1) * p.srcRow;
        const Pixel<T, C> p00 = LoadPx<T, C>(r0, sx), p01 = LoadPx<T, C>(r0, sx1);
        const Pixel<T, C> p10 = LoadPx<T, C>(r1, sx), p11 = LoadPx<T, C>(r1, sx1);
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            if constexpr (kFixedLinear<T>)
            {
                out.v[c] = BilinearQ15Scalar(p00.v[c], p01.v[c], p10.v[c], p11.v[c], FractionQ15(wx), FractionQ15(wy));
                continue;
            }
            float v;
            if constexpr (VARSHAPE)
            {
                v = (1.0f - wx) * ((float)p00.v[c] * (1.0f - wy) + (float)p10.v[c] * wy)
                  + wx * ((float)p01.v[c] * (1.0f - wy) + (float)p11.v[c] * wy);
            }
            else
            {
                v = (float)p00.v[c] * ((1.f - wx) * (1.f - wy)) + (float)p01.v[c] * (wx * (1.f - wy))
                  + (float)p10.v[c] * ((1.f - wx) * wy) + (float)p11.v[c] * (wx * wy);
            }
            out.v[c] = SaturateCast<T>(v);
        }
    }
    else if constexpr (INTERP == NVCV_INTERP_AREA)
    {
        // box filter over the source rectangle the output pixel covers, partial pixels weighted by
        // their covered fraction; taps outside the image read 0 (reference:
        // cuda_tools/InterpolationWrap.hpp:668-760, accumulation order kept)
        const float fsx1 = dx * scaleX, fsy1 = dy * scaleY;
        const float fsx2 = fsx1 + scaleX, fsy2 = fsy1 + scaleY;
        const int   xmin = (int)ceilf(fsx1), xmax = (int)floorf(fsx2);
        const int   ymin = (int)ceilf(fsy1), ymax = (int)floorf(fsy2);
        float       sum[C];
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            sum[c] = 0.f;
        }
        // pixels [xa, xb) of row y, each with weight w, in ascending order; what lies outside the image
        // contributes nothing, so the range is clipped once instead of testing every tap
        auto addRun = [&](int xa, int xb, int y, float w)
        {
            if (y < 0 || y >= p.srcH)
            {
                return;
            }
            // small pixels are fetched G at a time (one load of up to 16 bytes) and added in the same order
            constexpr int  PB  = (int)sizeof(Pixel<T, C>), G = PB <= 4 ? 4 : (PB <= 8 ? 2 : 1);
            const uint8_t *row = p.src + (int64_t)y * p.srcRow;
            xb                 = min(xb, p.srcW);
            int x              = max(xa, 0);
            if constexpr (G > 1)
            {
                for (; x + G <= xb; x += G)
                {
                    float t[G][C];
                    LoadTaps<T, C, G>(row, x * PB, y == p.srcH - 1, p.srcW * PB, t);
#pragma unroll
                    for (int k = 0; k < G; ++k)
                    {
#pragma unroll
                        for (int c = 0; c < C; ++c)
                        {
                            sum[c] += t[k][c] * w;
                        }
                    }
                }
            }
            for (; x < xb; ++x)
            {
                float t[1][C];
                LoadTaps<T, C, 1>(row, x * PB, y == p.srcH - 1, p.srcW * PB, t);
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    sum[c] += t[0][c] * w;
                }
            }
        };
        auto add = [&](int x, int y, float w) { addRun(x, x + 1, y, w); };
        // u8 pixels of 1, 3 or 4 channels at horizontal scales up to 2: the taps of one source row (a partial pixel on
        // the left, up to 2 whole ones, a partial one on the right) lie within 4 pixels, one load of 4 pixels instead
        // of one per tap (u8x3: a 2- and a 1-byte load per tap before; 226 -> 151 us per 32 x 1080p -> 720p). Which taps exist differs from lane to
        // lane, their order in the sums does not. The kernel is bound by the bytes its lanes ask for, not by
        // latency: with the windows of the 4 rows from ymin - 1 on all loaded before the first sum (4 loads
        // where 2 or 3 are needed) it took 208 us. Rows before the image's last one only: a load may read up
        // to 3 pixels past its taps.
        bool windowed = false;
        if constexpr (std::is_same_v<T, uint8_t> && (C == 1 || C == 3 || C == 4))
        {
            windowed = scaleX <= 2.f && p.srcW >= 4 && ymax < p.srcH - 1;
        }
        const bool hasLeft = xmin > fsx1, hasRight = xmax < fsx2;
        const int  winX = xmin - (hasLeft ? 1 : 0), innerN = min(xmax, p.srcW) - xmin, rightI = xmax - winX;
        [[maybe_unused]] auto loadWindow = [&](int y, uint32_t (&px)[4])
        {
            // 4 pixels of C bytes, pixel k to px[k] (channel c in byte c; higher bytes are not looked at)
            uint32_t w[C];
            LoadDwords<C>(p.src + (int64_t)y * p.srcRow + winX * C, w);
#pragma unroll
            for (int k = 0; k < 4; ++k)
            {
                if constexpr (C == 1)
                {
                    px[k] = w[0] >> (8 * k);
                }
                else if constexpr (C == 4)
                {
                    px[k] = w[k];
                }
                else
                {
                    px[k] = k == 0 ? w[0]
                          : k == 1 ? __builtin_amdgcn_alignbit(w[C > 1 ? 1 : 0], w[0], 24)
                          : k == 2 ? __builtin_amdgcn_alignbit(w[C > 2 ? 2 : 0], w[C > 1 ? 1 : 0], 16)
                                   : w[C > 2 ? 2 : 0] >> 8;
                }
            }
        };
        [[maybe_unused]] auto addPx = [&](uint32_t q, float w)
        {
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                sum[c] += (float)((q >> (8 * c)) & 0xFF) * w;
            }
        };
        [[maybe_unused]] auto addInner = [&](const uint32_t (&px)[4], float w) // pixels [xmin, xmax) of the row
        {
#pragma unroll
            for (int k = 0; k < 2; ++k)
            {
                if (k < innerN)
                {
                    addPx(hasLeft ? px[k + 1] : px[k], w);
                }
            }
        };
        [[maybe_unused]] auto addLeft  = [&](const uint32_t (&px)[4], float w) { addPx(px[0], w); }; // pixel xmin - 1
        [[maybe_unused]] auto addRight = [&](const uint32_t (&px)[4], float w)                        // pixel xmax
        {
            if (xmax < p.srcW)
            {
                addPx(rightI == 0 ? px[0] : rightI == 1 ? px[1] : rightI == 2 ? px[2] : px[3], w);
            }
        };
        // the rows between the partial ones: whole pixels, then the partial ones left and right
        [[maybe_unused]] auto addInnerRows = [&](float scale, bool partials)
        {
            for (int cy = ymin; cy < ymax; ++cy)
            {
                uint32_t px[4];
                loadWindow(cy, px);
                addInner(px, scale);
                if (partials && hasLeft)
                {
                    addLeft(px, (xmin - fsx1) * scale);
                }
                if (partials && hasRight)
                {
                    addRight(px, (fsx2 - xmax) * scale);
                }
            }
        };
        if (windowed && VARSHAPE && scaleX >= 1.0f && scaleY >= 1.0f)
        {
            const int iscaleX = SaturateCast<int32_t>(scaleX), iscaleY = SaturateCast<int32_t>(scaleY);
            if (scaleX == (float)iscaleX && scaleY == (float)iscaleY)
            {
                addInnerRows(1.f / (scaleX * scaleY), false);
            }
            else
            {
                // whole pixels of both partial rows, then the corners (top left, top right, bottom right, bottom left)
                const float scale = 1.f / (fminf(scaleX, p.srcW - fsx1) * fminf(scaleY, p.srcH - fsy1));
                addInnerRows(scale, true);
                uint32_t top[4] = {}, bot[4] = {};
                if (ymin > fsy1)
                {
                    loadWindow(ymin - 1, top);
                    addInner(top, (ymin - fsy1) * scale);
                }
                if (ymax < fsy2)
                {
                    loadWindow(ymax, bot);
                    addInner(bot, (fsy2 - ymax) * scale);
                }
                if (ymin > fsy1 && hasLeft)
                {
                    addLeft(top, (ymin - fsy1) * (xmin - fsx1) * scale);
                }
                if (ymin > fsy1 && hasRight)
                {
                    addRight(top, (ymin - fsy1) * (fsx2 - xmax) * scale);
                }
                if (ymax < fsy2 && hasRight)
                {
                    addRight(bot, (fsy2 - ymax) * (fsx2 - xmax) * scale);
                }
                if (ymax < fsy2 && hasLeft)
                {
                    addLeft(bot, (fsy2 - ymax) * (xmin - fsx1) * scale);
                }
            }
        }
        else if (windowed && !VARSHAPE)
        {
            if (ceilf(scaleX) == scaleX && ceilf(scaleY) == scaleY)
            {
                addInnerRows(1.f / (scaleX * scaleY), false);
            }
            else
            {
                const float scale = 1.f / (fminf(scaleX, p.srcW - fsx1) * fminf(scaleY, p.srcH - fsy1));
                addInnerRows(scale, true);
                if (ymin > fsy1)
                {
                    uint32_t px[4];
                    loadWindow(ymin - 1, px);
                    addInner(px, (ymin - fsy1) * scale);
                    if (hasLeft)
                    {
                        addLeft(px, (ymin - fsy1) * (xmin - fsx1) * scale);
                    }
                    if (hasRight)
                    {
                        addRight(px, (ymin - fsy1) * (fsx2 - xmax) * scale);
                    }
                }
                if (ymax < fsy2)
                {
                    uint32_t px[4];
                    loadWindow(ymax, px);
                    addInner(px, (fsy2 - ymax) * scale);
                    if (hasRight)
                    {
                        addRight(px, (fsy2 - ymax) * (fsx2 - xmax) * scale);
                    }
                    if (hasLeft)
                    {
                        addLeft(px, (fsy2 - ymax) * (xmin - fsx1) * scale);
                    }
                }
            }
        }
        else if constexpr (VARSHAPE)
        {
            // image batches follow the reference's separate kernel (legacy/resize_var_shape.cu:236-428):
            // same sums for reductions, corners added last; enlargements are a bilinear variant whose
            // fractions come from the inverse scale in double
            const int  iscaleX = SaturateCast<int32_t>(scaleX), iscaleY = SaturateCast<int32_t>(scaleY);
            const bool fast    = scaleX == (float)iscaleX && scaleY == (float)iscaleY;
            if (scaleX >= 1.0f && scaleY >= 1.0f)
            {
                if (fast)
                {
                    const float scale = 1.f / (scaleX * scaleY);
                    for (int cy = ymin; cy < ymax; ++cy)
                    {
                        addRun(xmin, xmax, cy, scale);
                    }
                }
                else
                {
                    const float scale = 1.f / (fminf(scaleX, p.srcW - fsx1) * fminf(scaleY, p.srcH - fsy1));
                    for (int cy = ymin; cy < ymax; ++cy)
                    {
                        addRun(xmin, xmax, cy, scale);
                        if (xmin > fsx1)
                        {
                            add(xmin - 1, cy, (xmin - fsx1) * scale);
                        }
                        if (xmax < fsx2)
                        {
                            add(xmax, cy, (fsx2 - xmax) * scale);
                        }
                    }
                    if (ymin > fsy1)
                    {
                        addRun(xmin, xmax, ymin - 1, (ymin - fsy1) * scale);
                    }
                    if (ymax < fsy2)
                    {
                        addRun(xmin, xmax, ymax, (fsy2 - ymax) * scale);
                    }
                    if (ymin > fsy1 && xmin > fsx1)
                    {
                        add(xmin - 1, ymin - 1, (ymin - fsy1) * (xmin - fsx1) * scale);
                    }
                    if (ymin > fsy1 && xmax < fsx2)
                    {
                        add(xmax, ymin - 1, (ymin - fsy1) * (fsx2 - xmax) * scale);
                    }
                    if (ymax < fsy2 && xmax < fsx2)
                    {
                        add(xmax, ymax, (fsy2 - ymax) * (fsx2 - xmax) * scale);
                    }
                    if (ymax < fsy2 && xmin > fsx1)
                    {
                        add(xmin - 1, ymax, (fsy2 - ymax) * (xmin - fsx1) * scale);
                    }
                }
            }
            else
            {
                const double invX = 1. / scaleX, invY = 1. / scaleY;
                int          sy = (int)floorf(dy * scaleY);
                float        fy = (float)((dy + 1) - (sy + 1) * invY);
                fy              = fy <= 0 ? 0.f : fy - (int)floorf(fy);
                int   sx = (int)floorf(dx * scaleX);
                float fx = (float)((dx + 1) - (sx + 1) * invX);
                fx       = fx < 0 ? 0.f : fx - (int)floorf(fx);
                if (sx < 0)
                {
                    fx = 0, sx = 0;
                }
                if (sx >= p.srcW - 1)
                {
                    fx = 0, sx = p.srcW - 2;
                }
                if (sy >= p.srcH - 1)
                {
                    sy = p.srcH - 2;
                }
                // sources of one row or column: the reference indexes outside the image; taps clamped here
                const int      x0 = max(sx, 0), x1 = min(sx + 1, p.srcW - 1), y0 = max(sy, 0), y1 = min(sy + 1, p.srcH - 1);
                const uint8_t *r0 = p.src + (int64_t)y0 * p.srcRow, *r1 = p.src + (int64_t)y1 * p.srcRow;
                const Pixel<T, C> p00 = LoadPx<T, C>(r0, x0), p10 = LoadPx<T, C>(r1, x0);
                const Pixel<T, C> p01 = LoadPx<T, C>(r0, x1), p11 = LoadPx<T, C>(r1, x1);
                const float       cx0 = 1.f - fx, cx1 = fx, cy0 = 1.f - fy, cy1 = fy;
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    sum[c] = (float)p00.v[c] * cx0 * cy0 + (float)p10.v[c] * cx0 * cy1 + (float)p01.v[c] * cx1 * cy0
                           + (float)p11.v[c] * cx1 * cy1;
                }
            }
        }
        else if (ceilf(scaleX) == scaleX && ceilf(scaleY) == scaleY)
        {
            const float scale = 1.f / (scaleX * scaleY);
            for (int cy = ymin; cy < ymax; ++cy)
            {
                addRun(xmin, xmax, cy, scale);
            }
        }
        else
        {
            const float scale = 1.f / (fminf(scaleX, p.srcW - fsx1) * fminf(scaleY, p.srcH - fsy1));
            for (int cy = ymin; cy < ymax; ++cy)
            {
                addRun(xmin, xmax, cy, scale);
                if (xmin > fsx1)
                {
                    add(xmin - 1, cy, (xmin - fsx1) * scale);
                }
                if (xmax < fsx2)
                {
                    add(xmax, cy, (fsx2 - xmax) * scale);
                }
            }
            if (ymin > fsy1)
            {
                addRun(xmin, xmax, ymin - 1, (ymin - fsy1) * scale);
                if (xmin > fsx1)
                {
                    add(xmin - 1, ymin - 1, (ymin - fsy1) * (xmin - fsx1) * scale);
                }
                if (xmax < fsx2)
                {
                    add(xmax, ymin - 1, (ymin - fsy1) * (fsx2 - xmax) * scale);
                }
            }
            if (ymax < fsy2)
            {
                addRun(xmin, xmax, ymax, (fsy2 - ymax) * scale);
                if (xmax < fsx2)
                {
                    add(xmax, ymax, (fsy2 - ymax) * (fsx2 - xmax) * scale);
                }
                if (xmin > fsx1)
                {
                    add(xmin - 1, ymax, (fsy2 - ymax) * (xmin - fsx1) * scale);
                }
            }
        }
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            out.v[c] = SaturateCast<T>(sum[c]);
        }
    }
    else // cubic
    {
        const float cx = (dx + .5f) * scaleX - .5f;
        const float cy = (dy + .5f) * scaleY - .5f;
        int         sx = (int)floorf(cx);
        int         sy = (int)floorf(cy);
        float       fx = cx - sx;
        const float fy = cy - sy;
        fx             = (sx < 1 || sx >= p.srcW - 3) ? 0.f : fx;
        sy             = max(1, min(sy, p.srcH - 3));
        sx             = max(1, min(sx, p.srcW - 3));
        float wx[4], wy[4];
        CubicCoeffs(fx, wx);
        CubicCoeffs(fy, wy);
        float sum[C];
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            sum[c] = 0.f;
        }
        [[maybe_unused]] int wq[4];
        if constexpr (kFixedCubic<T>)
        {
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                wx[i] *= 16384.f;
                wy[i] *= 1.f / 16384.f;
            }
            CubicWeightsQ14(wx, wq);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            // sources narrower/lower than 4 pixels: clamp the taps into the image
            const int      yy  = max(0, min(sy - 1 + j, p.srcH - 1));
            const uint8_t *row = p.src + (int64_t)yy * p.srcRow;
            Pixel<T, C>    t[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                t[i] = LoadPx<T, C>(row, max(0, min(sx - 1 + i, p.srcW - 1)));
            }
            if constexpr (kFixedCubic<T>)
            {
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    const int h = (int)t[0].v[c] * wq[0] + (int)t[1].v[c] * wq[1] + (int)t[2].v[c] * wq[2] + (int)t[3].v[c] * wq[3];
                    sum[c]      = j == 0 ? (float)h * wy[0] : fmaf((float)h, wy[j], sum[c]);
                }
                continue;
            }
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                if constexpr (VARSHAPE)
                {
                    sum[c] += wy[j]
                            * (wx[0] * (float)t[0].v[c] + wx[1] * (float)t[1].v[c] + wx[2] * (float)t[2].v[c]
                               + wx[3] * (float)t[3].v[c]);
                }
                else
                {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                    {
                        sum[c] += (float)t[i].v[c] * (wx[i] * wy[j]);
                    }
                }
            }
        }
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            out.v[c] = SaturateCast<T>(fabsf(sum[c]));
        }
    }
    return out;
}

template<class T, int C, int INTERP, bool VARSHAPE>
__device__ __forceinline__ void ResizePixel(const Plane &p, int dx, int dy)
{
    StorePx<T, C>(p.dst + (int64_t)dy * p.dstRow, dx, ResizeValue<T, C, INTERP, VARSHAPE>(p, dx, dy));
}

// The tile (in units of a wave's tile) of this wave in a launch of the tensor kernels below. Counted along the rows of tiles, a block
// writes and reads few long row pieces instead of many short ones, which the memory likes better, and only an image's last block has waves
// outside it, where many had as a block's four stood side by side (rows of 1024 pixels and more) or below one another. us
// as they stood / counted along the rows: bicubic u8x3 182 x 219 x 77 -> 593 x 209 41.6 / 28.7, 101 x 241 x 274 -> 572 x 655 56.3 / 42.9, 40 x 300 x 300 -> 600 x
// 600 24.6 / 21.8, 32 x 720p -> 1080p 90.1 / 86.4; u8x4 40 x 300 x 300 -> 600 x 600 22.7 / 20.5; nearest neighbour u8x4 200 x 86 x 80 -> 307 x 287 22.5 / 18.3,
// u8x3 50 x 209 x 770 -> 362 x 1335 25.2 / 19.5; box filter u8x3 4 x 3146 x 1185 -> 1646 x 620 25.5 / 20.6, u8x1 171 x 1723 x 388 -> 609 x 137 65.7 / 57.3; wave
// patches, bilinear u8x3 193 x 171 x 925 -> 68 x 367 30.9 / 26.9, u8x4 12 x 702 x 2707 -> 466 x 1447 26.5 / 22.7. Means over 280 to 490 random launches each, inputs in and out of
// the memory's cache: nearest neighbour u8x4 0.92 and 0.94, f32x1 0.91 and 0.93, bicubic u8x1 and u8x4 0.96 and 0.97, f32x1 0.94 and 0.95, box filter 0.97 to 0.99.
// Single launches lose in all of these, u8x4 nearest neighbour among them that starts rows with a block no more: 37 x 572 x 202 -> 1707 x 622 39.7 / 43.0, 39 x 899 x 224 -> 1983 x 447
// 34.3 / 37.4, but 72 x 1402 x 50 -> 3280 x 117 26.1 / 21.3, 15 x 1101 x 195 -> 3632 x 646 28.5 / 26.0, 65 of these 0.99 in the mean. Not counted so: the bilinear strips of
// 8-bit pixels whose rows are short (u8x3 80 x 650 x 104 -> 1274 x 195 24.0 / 29.5, u8x4 190 x 307 x 16 -> 942 x 50 14.9 / 16.7; those of
// 1024 pixels and more that fill blocks to 80 % are: FlatBlocks), rows that share what they read (SharedRowsPay), the bicubic strips of four floats and of
// few waves, one-pixel waves of bilinear and bicubic and the staged bicubic below vertical scales of 2 and 4: beside their launches.
__device__ __forceinline__ WaveTile WaveTileOf(const WaveOrder &order)
{
    // (the wave's number as a scalar: tile origins, row terms and loop counters then stay on the scalar unit)
    return TileOfWave(order, blockIdx.x, blockIdx.y, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), blockDim.x >> 6);
}

static inline bool FlatBlocks(int dstW, int waveW)
{
    const int64_t span = 4 * (int64_t)waveW;
    return dstW >= 1024 && DivUp(dstW, (int)span) * span * 4 <= (int64_t)dstW * 5;
}

// Whether the source pixels that the output rows of a stacked block need not fetch again, because the row above has, are `of` / `in` of the
// pixels written or more, the rows fill their waves of waveW x waveH to `full` per cent and the columns their blocks of four to 3/4 (6909 x 211 x 2 f32x1 bicubic ->
// 107 x 17, one row in a second block of 16: 46.8 us along the rows, 68.7 below one another). Such launches lose along the rows, where blocks on all XCDs fetch a source row for
// the output rows that it serves: as many of them as rows, up to 8. So they do not where the source has less than 1 / `times` of the pixels written,
// which 8 caches take little time to fetch (the more output rows to a source row, the wider the sources that still lose). Time over that along the rows, 1000 to 1900
// random launches of each form enlarged 1.3 to 90 times, inputs in the memory's cache, with sources and columns of any size / so: nearest neighbour 0.84 / 0.79, bilinear u8x4
// 0.94 / 0.93, bicubic f32x3 1.02 / 0.99, f32x1 0.85 / 0.86, the slowest of it 1.47 / 1.26. Just outside `times` nearest neighbour takes 1.03 to 1.14 below one another, u8x4 1.04 to
// 1.09, f32x3 1.03, f32x1 1.02 to 1.07.
static inline bool SharedRowsPay(const ResizeArgs &a, int waveW, int waveH, int in, int of, int times, int full = 80)
{
    return in * (int64_t)(a.dstH - a.srcH) * a.srcW >= of * (int64_t)a.dstW * a.dstH
        && times * (int64_t)a.srcW * a.srcH >= (int64_t)a.dstW * a.dstH
        && full * (int64_t)DivUp(a.dstW, waveW) * waveW <= 100 * (int64_t)a.dstW && 3 * (int64_t)DivUp(a.dstH, 4 * waveH) * 4 * waveH <= 4 * (int64_t)a.dstH;
}

// Grid of a launch whose waves own tiles of waveW x waveH.
static inline dim3 WaveTileGrid(int dstW, int dstH, int N, int waveW, int waveH, const WaveOrder &order, int waves = 4)
{
    const WaveBlocks blocks = BlocksOfWaves(dstW, dstH, waveW, waveH, order, waves);
    return dim3(blocks.x, blocks.y, N);
}

template<class T, int C, int INTERP>
__global__ __launch_bounds__(256) void ResizeTensorKernel(const ResizeArgs a, const WaveOrder order)
{
    // (the wave's number as a vector here, where a wave is one pixel per lane: with scalar places the store's address waits for the scalar unit. Nearest
    // neighbour f32x3 19 x 1750 x 278 -> 826 x 706 47.5 us, so 44.2, 2 x 1636 x 1610 -> 1433 x 4096 48.5 and 44.1, others 0.98 to 1.00. Not for box sums, whose
    // loops over rows the scalar unit counts: u8x1 1.07 times slower in the mean of 134 launches as a vector, 3 x 2106 x 1884 -> 12 x 27 418 and 492, u8x3 1.03, f32x1
    // 1.04; of three and four floats 0.99, u8x4 1.00)
    constexpr bool kScalar = INTERP == NVCV_INTERP_AREA && sizeof(Pixel<T, C>) <= 4;
    const WaveTile t  = kScalar ? WaveTileOf(order) : TileOfWave(order, blockIdx.x, blockIdx.y, threadIdx.x >> 6, 4);
    const int      dx = t.x * kTileW + (threadIdx.x & 63), dy = t.y;
    if (dx >= a.dstW || dy >= a.dstH)
    {
        return;
    }
    const Plane p = GetPlanes<false>(a, blockIdx.z);
    ResizePixel<T, C, INTERP, false>(p, dx, dy);
}

template<class T, int C, int INTERP>
__global__ __launch_bounds__(256) void ResizeVarShapeKernel(const ResizeArgs a, const VarTiles tiles)
{
    const TileCoord tc = LocateTile(tiles, blockIdx.x);
    const Plane     p  = GetPlanes<true>(a, tc.image);
    const int       dx = tc.tx * kTileW + (threadIdx.x & 63);
    const int       dy = tc.ty * kTileH + (threadIdx.x >> 6);
    if (dx >= p.dstW || dy >= p.dstH)
    {
        return;
    }
    ResizePixel<T, C, INTERP, true>(p, dx, dy);
}

// ---------------------------------------------------------------------------------------------
// Wave-patch form for small pixels. The per-pixel form above issues one load per tap and one store
// per channel (8 tap loads and 3 byte stores per u8x3 bilinear pixel) and is bound by the number of
// memory instructions, not by bytes or arithmetic. Here the horizontally adjacent taps of a sample
// (2 for bilinear, 4 for bicubic) come from one load, and lanes exchange results so that each
// stores 4 consecutive pixels as whole dwords. Arithmetic: the expressions of ResizeValue, term for
// term.

// Per-column and per-row terms of a sample: source index and weights, the expressions of
// ResizeValue. W = number of weights (0 nearest, 1 linear, 4 cubic); sources are >= 4 pixels wide.
template<int W>
struct AxisTerms
{
    int   s;                // nearest: source index; linear: first tap; cubic: second tap
    float w[W > 0 ? W : 1]; // linear: weight of the second tap
};

template<int INTERP>
constexpr int kWeights = INTERP == NVCV_INTERP_NEAREST ? 0 : (INTERP == NVCV_INTERP_LINEAR ? 1 : 4);

template<int INTERP>
__device__ __forceinline__ AxisTerms<kWeights<INTERP>> Axis(float scale, int d, int srcSize)
{
    AxisTerms<kWeights<INTERP>> a;
    if constexpr (INTERP == NVCV_INTERP_NEAREST)
    {
        a.s = min((int)floorf(scale * (d + 0.5f)), srcSize - 1);
    }
    else if constexpr (INTERP == NVCV_INTERP_LINEAR)
    {
        const float f = (d + .5f) * scale - .5f;
        const int   s = (int)floorf(f);
        a.w[0]        = (s < 0) ? 0.f : ((s > srcSize - 2) ? 1.f : f - s);
        a.s           = max(0, min(s, srcSize - 2));
    }
    else
    {
        const float c = (d + .5f) * scale - .5f;
        const int   s = (int)floorf(c);
        float       f = c - s;
        a.s           = s;
        a.w[0]        = f; // finished by the caller: the two axes treat the fraction differently
    }
    return a;
}

// Lane `from` (constant) of every field, as wave-uniform values.
template<int W>
__device__ __forceinline__ AxisTerms<W> FromLane(const AxisTerms<W> &a, int from)
{
    AxisTerms<W> r;
    r.s = __builtin_amdgcn_readlane(a.s, from);
#pragma unroll
    for (int i = 0; i < (W > 0 ? W : 1); ++i)
    {
        r.w[i] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(a.w[i]), from));
    }
    return r;
}

__device__ __forceinline__ float ReadLane(float v, int lane)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// The 8-bit bicubic sum of one output pixel per lane: rows y0 .. y0 + 3 (clamped into the image), their windows of 4
// pixels at `at` + `shift`, the packed horizontal weights and the vertical ones times 2^-14 (wave-uniform). All four
// windows are requested before the first sum.
template<int C, bool GUARDED, bool ODD>
__device__ __forceinline__ uint32_t CubicRowsQ14(const Plane &p, int y0, uint32_t at, uint32_t shift, uint32_t rowBytes,
                                                 uint32_t w01, uint32_t w23, const float (&wy)[4])
{
    uint32_t       r[4][C];
    const uint8_t *first = p.src + (int64_t)y0 * p.srcRow;
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        const int      yy   = GUARDED ? max(0, min(y0 + j, p.srcH - 1)) : y0 + j;
        const uint8_t *line = GUARDED ? p.src + (int64_t)yy * p.srcRow : first + (int64_t)j * p.srcRow;
        LoadQuadWindow<C, GUARDED, ODD>(line, at, shift, yy == p.srcH - 1, rowBytes, r[j]);
    }
    float acc[C];
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        const float w = wy[j];
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            const float h = RowSumQ14(QuadTapPair<C>(r[j], 0, c), QuadTapPair<C>(r[j], 2, c), w01, w23);
            acc[c]        = j == 0 ? h * w : fmaf(h, w, acc[c]);
        }
    }
    uint32_t q = 0;
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        q = __builtin_amdgcn_cvt_pk_u8_f32(fabsf(acc[c]), c, q);
    }
    return q;
}

// The same for TWO vertically adjacent output pixels per lane whose 4-row windows start `N - 4` rows apart (0 .. 2) and
// lie inside the image, clear of its last row: the N source rows from y0 on are loaded once, each row's sums are
// formed once, and each pixel adds its own four in ascending order - the sums and their order are those of
// CubicRowsQ14, so the result is the same bit for bit. At scale 1.5 that is 5 or 6 row sums where two pixels took 8.
template<int C, int N, bool ODD>
__device__ __forceinline__ void CubicRowPairQ14(const Plane &p, int y0, uint32_t at, uint32_t shift, uint32_t rowBytes,
                                                uint32_t w01, uint32_t w23, const float (&wyA)[4], const float (&wyB)[4],
                                                uint32_t (&out)[2])
{
    uint32_t       r[N][C];
    const uint8_t *first = p.src + (int64_t)y0 * p.srcRow;
#pragma unroll
    for (int j = 0; j < N; ++j)
    {
        LoadQuadWindow<C, false, ODD>(first + (int64_t)j * p.srcRow, at, shift, false, rowBytes, r[j]);
    }
    float accA[C], accB[C];
#pragma unroll
    for (int j = 0; j < N; ++j)
    {
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            const float h = RowSumQ14(QuadTapPair<C>(r[j], 0, c), QuadTapPair<C>(r[j], 2, c), w01, w23);
            if (j < 4)
            {
                accA[c] = j == 0 ? h * wyA[0] : fmaf(h, wyA[j], accA[c]);
            }
            if (j >= N - 4)
            {
                accB[c] = j == N - 4 ? h * wyB[0] : fmaf(h, wyB[j - (N - 4)], accB[c]);
            }
        }
    }
    out[0] = out[1] = 0;
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        out[0] = __builtin_amdgcn_cvt_pk_u8_f32(fabsf(accA[c]), c, out[0]);
        out[1] = __builtin_amdgcn_cvt_pk_u8_f32(fabsf(accB[c]), c, out[1]);
    }
}

// The part of the 8-bit bicubic sum that depends on the output column only.
struct CubicColumnQ14
{
    uint32_t w01, w23;  // horizontal weights in units of 2^-14, packed in pairs
    uint32_t at, shift; // the window load's byte offset in a row and the window's position in it
};

template<int C>
__device__ __forceinline__ CubicColumnQ14 CubicColumn(const AxisTerms<4> &col)
{
    CubicColumnQ14 q;
    float          wx[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        wx[i] = col.w[i] * 16384.f;
    }
    CubicWeightPairsQ14(wx, q.w01, q.w23);
    const uint32_t off = (uint32_t)(col.s - 1) * C;
    q.at               = C == 4 ? off : off & ~3u;
    q.shift            = off & 3u;
    return q;
}

// A lane's 4 output pixels (rows k = 0 .. 3 of a wave patch, row terms in lanes 0 .. 3 of `rows`, vertical weights
// already in units of 2^-14) of the 8-bit bicubic form, clear of the image's last row: output rows in pairs that
// share the source rows between their windows (wave-uniform choice by how far the windows are apart; farther than
// 2: one by one).
template<int C, bool ODD>
__device__ __forceinline__ void CubicPatchPairsQ14(const Plane &p, const AxisTerms<4> &col, const AxisTerms<4> &rows,
                                                   uint32_t (&q)[4])
{
    const CubicColumnQ14 cq = CubicColumn<C>(col);
    const uint32_t       rb = (uint32_t)p.srcW * C;
#pragma unroll
    for (int k = 0; k < 4; k += 2)
    {
        const auto rowA = FromLane(rows, k), rowB = FromLane(rows, k + 1);
        const int  apart = rowB.s - rowA.s;
        uint32_t   two[2];
        if (apart == 1)
        {
            CubicRowPairQ14<C, 5, ODD>(p, rowA.s - 1, cq.at, cq.shift, rb, cq.w01, cq.w23, rowA.w, rowB.w, two);
        }
        else if (apart == 2)
        {
            CubicRowPairQ14<C, 6, ODD>(p, rowA.s - 1, cq.at, cq.shift, rb, cq.w01, cq.w23, rowA.w, rowB.w, two);
        }
        else if (apart == 0)
        {
            CubicRowPairQ14<C, 4, ODD>(p, rowA.s - 1, cq.at, cq.shift, rb, cq.w01, cq.w23, rowA.w, rowB.w, two);
        }
        else
        {
            two[0] = CubicRowsQ14<C, false, ODD>(p, rowA.s - 1, cq.at, cq.shift, rb, cq.w01, cq.w23, rowA.w);
            two[1] = CubicRowsQ14<C, false, ODD>(p, rowB.s - 1, cq.at, cq.shift, rb, cq.w01, cq.w23, rowB.w);
        }
        q[k]     = two[0];
        q[k + 1] = two[1];
    }
}

// One output pixel from its column terms (per lane) and row terms (wave-uniform). GUARDED: the image's last row may
// be among the rows read, so every tap load tests for it (its loads must not run past the image's end); the caller
// settles that once per wave patch, because a wave-uniform test in front of a load keeps the compiler from requesting
// the next load before this one has returned.
template<class T, int C, int INTERP, bool VARSHAPE, bool GUARDED, bool ODD>
__device__ __forceinline__ Pixel<T, C> SampleWide(const Plane &p, const AxisTerms<kWeights<INTERP>> &col,
                                                  const AxisTerms<kWeights<INTERP>> &row)
{
    constexpr int PB       = sizeof(Pixel<T, C>);
    const int     rowBytes = p.srcW * PB;
    Pixel<T, C>   out;
    if constexpr (INTERP == NVCV_INTERP_NEAREST)
    {
        float t[1][C];
        LoadTaps<T, C, 1>(p.src + (int64_t)row.s * p.srcRow, col.s * PB, GUARDED && row.s == p.srcH - 1, rowBytes, t);
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            out.v[c] = (T)t[0][c]; // exact: the value came from a T
        }
    }
    else if constexpr (INTERP == NVCV_INTERP_LINEAR)
    {
        const int   y0 = row.s, y1 = min(row.s + 1, p.srcH - 1);
        const float wx = col.w[0], wy = row.w[0];
        if constexpr (kFixedLinear<T>)
        {
            uint32_t r0[2], r1[2], top, bottom, q = 0;
            LoadTapPairBytes<C>(p.src + (int64_t)y0 * p.srcRow, col.s * PB, GUARDED && y0 == p.srcH - 1, rowBytes, r0);
            LoadTapPairBytes<C>(p.src + (int64_t)y1 * p.srcRow, col.s * PB, GUARDED && y1 == p.srcH - 1, rowBytes, r1);
            WeightPairsQ15(FractionQ15(wx), FractionQ15(wy), top, bottom);
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                const uint32_t sel = 0x0c000c00u | (uint32_t)c | ((uint32_t)(c + C) << 16);
                q = BlendQ15(__builtin_amdgcn_perm(r0[1], r0[0], sel), __builtin_amdgcn_perm(r1[1], r1[0], sel), top, bottom, c, q);
            }
            __builtin_memcpy(&out, &q, PB);
            return out;
        }
        float       t0[2][C], t1[2][C];
        LoadTaps<T, C, 2>(p.src + (int64_t)y0 * p.srcRow, col.s * PB, GUARDED && y0 == p.srcH - 1, rowBytes, t0);
        LoadTaps<T, C, 2>(p.src + (int64_t)y1 * p.srcRow, col.s * PB, GUARDED && y1 == p.srcH - 1, rowBytes, t1);
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            float v;
            if constexpr (VARSHAPE)
            {
                v = (1.0f - wx) * (t0[0][c] * (1.0f - wy) + t1[0][c] * wy)
                  + wx * (t0[1][c] * (1.0f - wy) + t1[1][c] * wy);
            }
            else
            {
                v = t0[0][c] * ((1.f - wx) * (1.f - wy)) + t0[1][c] * (wx * (1.f - wy)) + t1[0][c] * ((1.f - wx) * wy)
                  + t1[1][c] * (wx * wy);
            }
            out.v[c] = SaturateCast<T>(v);
        }
    }
    else if constexpr (kFixedCubic<T>)
    {
        // (the column's part of this does not depend on the row and is computed once per lane)
        const CubicColumnQ14 cq = CubicColumn<C>(col);
        // rows row.s - 1 .. row.s + 2, inside the image for sources of 4 rows and more; four windows together
        const uint32_t q = CubicRowsQ14<C, GUARDED, ODD>(p, row.s - 1, cq.at, cq.shift, (uint32_t)rowBytes, cq.w01, cq.w23, row.w);
        __builtin_memcpy(&out, &q, PB);
    }
    else
    {
        float sum[C];
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            sum[c] = 0.f;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            const int yy = max(0, min(row.s - 1 + j, p.srcH - 1));
            float     t[4][C];
            LoadTaps<T, C, 4>(p.src + (int64_t)yy * p.srcRow, (col.s - 1) * PB, GUARDED && yy == p.srcH - 1, rowBytes, t);
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                if constexpr (VARSHAPE)
                {
                    sum[c] += row.w[j] * (col.w[0] * t[0][c] + col.w[1] * t[1][c] + col.w[2] * t[2][c] + col.w[3] * t[3][c]);
                }
                else
                {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                    {
                        sum[c] += t[i][c] * (col.w[i] * row.w[j]);
                    }
                }
            }
        }
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            out.v[c] = SaturateCast<T>(fabsf(sum[c]));
        }
    }
    return out;
}

// Column (horizontal == true) or row terms of output index d, finished for sampling.
template<int INTERP>
__device__ __forceinline__ AxisTerms<kWeights<INTERP>> FinishedAxis(float scale, int d, int srcSize, bool horizontal)
{
    AxisTerms<kWeights<INTERP>> a = Axis<INTERP>(scale, d, srcSize);
    if constexpr (INTERP == NVCV_INTERP_CUBIC)
    {
        // the reference zeroes the horizontal fraction next to the image border, not the vertical one
        float f = a.w[0];
        f       = (horizontal && (a.s < 1 || a.s >= srcSize - 3)) ? 0.f : f;
        a.s     = max(1, min(a.s, srcSize - 3));
        CubicCoeffs(f, a.w);
    }
    return a;
}

// Stores a wave's 64-column x 4-row patch at (x0, y0): q[d][k] is dword d of the pixel (x0 + lane, y0 + k). After
// the 4x4 transposes lane l owns row y0 + (l & 3), columns x0 + 4 * (l >> 2) .. + 3, written as whole dwords.
template<class T, int C>
__device__ __forceinline__ void StoreWavePatch(const Plane &p, int x0, int y0, int lane,
                                               uint32_t (&q)[(sizeof(Pixel<T, C>) + 3) / 4][4])
{
    constexpr int PB = sizeof(Pixel<T, C>), D = (PB + 3) / 4;
#pragma unroll
    for (int d = 0; d < D; ++d)
    {
        QuadTranspose(q[d], lane & 3);
    }
    const int dy = y0 + (lane & 3), dx0 = x0 + 4 * (lane >> 2);
    if (dy >= p.dstH || dx0 >= p.dstW)
    {
        return;
    }
    uint8_t *to = p.dst + (int64_t)dy * p.dstRow + (int64_t)dx0 * PB;

    if (dx0 + 4 <= p.dstW)
    {
        uint32_t w[PB];
        PackQuad<PB>(q, w);
        StoreDwordsNT<PB>(to, w);
    }
    else
    {
#pragma unroll
        for (int k = 0; k < 3; ++k)
        {
            if (dx0 + k < p.dstW)
            {
                uint32_t w[D];
#pragma unroll
                for (int d = 0; d < D; ++d)
                {
                    w[d] = q[d][k];
                }
                Pixel<T, C> px;
                __builtin_memcpy(&px, w, PB);
                reinterpret_cast<Pixel<T, C> *>(to)[k] = px;
            }
        }
    }
}

// One wave resizes a 64-column x 4-row patch of the output whose top left pixel is (x0, y0), both
// wave-uniform. Sampling: lane l owns column x0 + l and computes its 4 rows (the column terms are
// shared; neighbouring lanes read neighbouring source pixels whatever the scale). Storing: after
// the 4x4 transposes lane l owns row y0 + (l & 3), columns x0 + 4 * (l >> 2) .. + 3.
template<class T, int C, int INTERP, bool VARSHAPE, bool ODD = false>
__device__ __forceinline__ void ResizeWavePatch(const Plane &p, int x0, int y0)
{
    constexpr int PB = sizeof(Pixel<T, C>), D = (PB + 3) / 4;
    if (x0 >= p.dstW || y0 >= p.dstH)
    {
        return;
    }
    const int   lane   = threadIdx.x & 63;
    const float scaleX = p.scaleX, scaleY = p.scaleY;
    // uniform per image (the 8-bit bicubic form loads whole dwords around 4 pixels: rows of 16 bytes or more, 8 for
    // one channel)
    const bool wide = p.srcW >= 4 && (INTERP != NVCV_INTERP_CUBIC || !kFixedCubic<T> || p.srcW * C >= (C == 1 ? 8 : 16));
    // columns and rows past the output compute a duplicate of the last one: every lane takes part in
    // the transposes
    const int dx = min(x0 + lane, p.dstW - 1);
    uint32_t  q[D][4];
    if (wide)
    {
        const auto col = FinishedAxis<INTERP>(scaleX, dx, p.srcW, true);
        // the 4 rows' terms are computed side by side (lane l: row l & 3) and then read as uniform values
        auto rows = FinishedAxis<INTERP>(scaleY, min(y0 + (lane & 3), p.dstH - 1), p.srcH, false);
        if constexpr (INTERP == NVCV_INTERP_CUBIC && kFixedCubic<T>)
        {
            // the vertical weights go with row sums in units of 2^-14
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                rows.w[i] *= 1.f / 16384.f;
            }
        }
        // the last source row the patch reads (row indices ascend with the output row; bilinear reads one more, bicubic
        // two): only a patch that reaches the image's last row needs the guarded loads (wave-uniform)
        constexpr int reach = INTERP == NVCV_INTERP_NEAREST ? 0 : (INTERP == NVCV_INTERP_LINEAR ? 1 : 2);
        auto          sample = [&](auto guarded)
        {
#pragma unroll
            for (int k = 0; k < 4; ++k)
            {
                const Pixel<T, C> out  = SampleWide<T, C, INTERP, VARSHAPE, decltype(guarded)::value, ODD>(p, col, FromLane(rows, k));
                uint32_t          w[D] = {};
                __builtin_memcpy(w, &out, PB);
#pragma unroll
                for (int d = 0; d < D; ++d)
                {
                    q[d][k] = w[d];
                }
            }
        };
        if (__builtin_amdgcn_readlane(rows.s, 3) + reach >= p.srcH - 1)
        {
            sample(std::true_type{});
        }
        else if constexpr (INTERP == NVCV_INTERP_CUBIC && kFixedCubic<T>)
        {
            CubicPatchPairsQ14<C, ODD>(p, col, rows, q[0]);
        }
        else
        {
            sample(std::false_type{});
        }
    }
    else
    {
#pragma unroll 1
        for (int k = 0; k < 4; ++k)
        {
            const Pixel<T, C> out  = ResizeValue<T, C, INTERP, VARSHAPE>(p, dx, min(y0 + k, p.dstH - 1));
            uint32_t          w[D] = {};
            __builtin_memcpy(w, &out, PB);
#pragma unroll
            for (int d = 0; d < D; ++d)
            {
                q[d][0] = k == 0 ? w[d] : q[d][0];
                q[d][1] = k == 1 ? w[d] : q[d][1];
                q[d][2] = k == 2 ? w[d] : q[d][2];
                q[d][3] = k == 3 ? w[d] : q[d][3];
            }
        }
    }
    StoreWavePatch<T, C>(p, x0, y0, lane, q);
}

// 8-bit bilinear at horizontal scales up to 2. The cost of the wave-patch form there is the number
// of tap loads (the texture addresser is busy 76-90 % of the time). The taps of two neighbouring
// output columns lie within 4 source pixels, so here a lane owns 2 columns x 2 rows and fetches each
// source row once for both columns (one 4-, 12- or 16-byte load): half the loads. A wave covers 128
// columns x 2 rows; lanes 2j and 2j+1 then swap a pixel pair each, so that lane 2j stores columns
// 4j .. 4j+3 of the first row and lane 2j+1 those of the second. Arithmetic as in SampleWide.
// Pixels travel as one dword each (channel c in byte c; higher bytes are don't-care).
template<int C>
struct __attribute__((packed, aligned(1))) TapWindow
{
    uint32_t w[C]; // 4 pixels of C bytes
};

// Pixel k (0 .. 3) of a window.
template<int C>
__device__ __forceinline__ uint32_t WindowPixel(const TapWindow<C> &t, int k)
{
    if constexpr (C == 4)
    {
        return t.w[k];
    }
    else if constexpr (C == 1)
    {
        return t.w[0] >> (8 * k);
    }
    else
    {
        static_assert(C == 3);
        return k == 0 ? t.w[0]
             : k == 1 ? __builtin_amdgcn_alignbit(t.w[1], t.w[0], 24)
             : k == 2 ? __builtin_amdgcn_alignbit(t.w[2], t.w[1], 16)
                      : t.w[2] >> 8;
    }
}

// The 4 pixels that start at `at` (rows before the image's last one only: the load may read past the row), in two
// steps so that a caller can request several windows before it touches the first.
// u8x3: the aligned 16 bytes that hold the window's 12, funnel-shifted into place. The texture path takes a
// 12-byte load that is not dword aligned apart into about three times as many cache accesses (counters:
// 63 against 20 per wave-load), and these kernels wait for that unit: 1080p -> 720p 61.5 -> 59.9 us,
// 720p -> 1080p 117 -> 101 us. Reads at most 3 bytes before and 4 after the window.
template<int C>
struct RawTapWindow
{
    uint32_t d[C == 3 ? 4 : C];
    uint32_t mis;
};

template<int C>
__device__ __forceinline__ RawTapWindow<C> RequestTapWindow(const uint8_t *at)
{
    RawTapWindow<C> r;
    if constexpr (C == 3)
    {
        struct alignas(4) W4
        {
            uint32_t d[4];
        };
        r.mis      = (uint32_t)reinterpret_cast<uintptr_t>(at) & 3u;
        const W4 w = *reinterpret_cast<const W4 *>(at - r.mis);
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            r.d[i] = w.d[i];
        }
    }
    else
    {
        r.mis                = 0;
        const TapWindow<C> t = *reinterpret_cast<const TapWindow<C> *>(at);
#pragma unroll
        for (int i = 0; i < C; ++i)
        {
            r.d[i] = t.w[i];
        }
    }
    return r;
}

template<int C>
__device__ __forceinline__ TapWindow<C> FinishTapWindow(const RawTapWindow<C> &r)
{
    TapWindow<C> t;
    if constexpr (C == 3)
    {
        t.w[0] = __builtin_amdgcn_alignbyte(r.d[1], r.d[0], r.mis);
        t.w[1] = __builtin_amdgcn_alignbyte(r.d[2], r.d[1], r.mis);
        t.w[2] = __builtin_amdgcn_alignbyte(r.d[3], r.d[2], r.mis);
    }
    else
    {
#pragma unroll
        for (int i = 0; i < C; ++i)
        {
            t.w[i] = r.d[i];
        }
    }
    return t;
}

template<int C>
__device__ __forceinline__ TapWindow<C> LoadTapWindowAt(const uint8_t *at)
{
    return FinishTapWindow<C>(RequestTapWindow<C>(at));
}

template<int C>
__device__ __forceinline__ TapWindow<C> LoadTapWindow(const Plane &p, int y, int xs)
{
    return LoadTapWindowAt<C>(p.src + (int64_t)y * p.srcRow + xs * C);
}

// One pixel from its four taps (a dword each, channel c in byte c) and the float32 weights of the second taps.
template<int C>
__device__ __forceinline__ uint32_t BilinearU8(uint32_t p00, uint32_t p01, uint32_t p10, uint32_t p11, float wx, float wy)
{
    return BilinearQ15<C>(p00, p01, p10, p11, FractionQ15(wx), FractionQ15(wy));
}

template<int C, bool VARSHAPE>
__device__ __forceinline__ void ResizeLinearPairsU8(const Plane &p, int x0, int y0)
{
    if (x0 >= p.dstW || y0 >= p.dstH)
    {
        return;
    }
    const int  lane = threadIdx.x & 63;
    const bool odd  = (lane & 1) != 0;
    // columns and rows past the output compute a duplicate of the last one: every lane takes part in the swap
    const auto colA  = Axis<NVCV_INTERP_LINEAR>(p.scaleX, min(x0 + 2 * lane, p.dstW - 1), p.srcW);
    const auto colB  = Axis<NVCV_INTERP_LINEAR>(p.scaleX, min(x0 + 2 * lane + 1, p.dstW - 1), p.srcW);
    const int  delta = colB.s - colA.s; // 0 .. 2 at scales up to 2
    // the 2 rows' terms are computed side by side (even lanes the first, odd lanes the second)
    const auto rows = Axis<NVCV_INTERP_LINEAR>(p.scaleY, min(y0 + (lane & 1), p.dstH - 1), p.srcH);
    uint32_t   pxA[2], pxB[2];
    const auto row0 = FromLane(rows, 0), row1 = FromLane(rows, 1);
    // taps of source row y for both columns: A's two, then B's
    auto fetchLast = [&](int y, uint32_t (&t)[4]) // the image's last row: nothing may be read past its end
    {
        const uint8_t *line = p.src + (int64_t)y * p.srcRow;
        float          a[2][C], b[2][C];
        LoadTaps<uint8_t, C, 2>(line, colA.s * C, true, p.srcW * C, a);
        LoadTaps<uint8_t, C, 2>(line, colB.s * C, true, p.srcW * C, b);
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            t[i] = 0;
        }
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            t[0] |= (uint32_t)a[0][c] << (8 * c);
            t[1] |= (uint32_t)a[1][c] << (8 * c);
            t[2] |= (uint32_t)b[0][c] << (8 * c);
            t[3] |= (uint32_t)b[1][c] << (8 * c);
        }
    };
    auto window = [&](int y) { return LoadTapWindow<C>(p, y, colA.s); };
    auto unpack = [&](const TapWindow<C> &win, uint32_t (&t)[4])
    {
        const uint32_t k0 = WindowPixel<C>(win, 0), k1 = WindowPixel<C>(win, 1), k2 = WindowPixel<C>(win, 2),
                       k3 = WindowPixel<C>(win, 3);
        t[0] = k0;
        t[1] = k1;
        t[2] = delta == 0 ? k0 : (delta == 1 ? k1 : k2);
        t[3] = delta == 0 ? k1 : (delta == 1 ? k2 : k3);
    };
    const int ya0 = row0.s, yb0 = min(row0.s + 1, p.srcH - 1), ya1 = row1.s, yb1 = min(row1.s + 1, p.srcH - 1);
    uint32_t  top[2][4], bot[2][4];
    if (max(yb0, yb1) < p.srcH - 1) // wave-uniform; the usual case: all four window loads go out together
    {
        // All four windows are requested before anything else (a load behind one of the tests below would wait for
        // the loads before it); the two output rows often share source rows (always when enlarging), whose taps
        // are taken apart once.
        auto request = [&](int y) { return RequestTapWindow<C>(p.src + (int64_t)y * p.srcRow + colA.s * C); };
        const RawTapWindow<C> r0 = request(ya0), r1 = request(yb0), r2 = request(ya1), r3 = request(yb1);
        // a use the compiler cannot move (without it the last two loads sink into the branches that need them) behind
        // a line the instruction scheduler does not cross (or it starts on the first window between the loads)
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::"v"(r0.d[0]), "v"(r1.d[0]), "v"(r2.d[0]), "v"(r3.d[0]));
        const TapWindow<C> w0 = FinishTapWindow<C>(r0), w1 = FinishTapWindow<C>(r1), w2 = FinishTapWindow<C>(r2),
                           w3 = FinishTapWindow<C>(r3);
        unpack(w0, top[0]);
        unpack(w1, bot[0]);
        if (ya1 == ya0)
        {
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                top[1][i] = top[0][i];
                bot[1][i] = bot[0][i];
            }
        }
        else
        {
            if (ya1 == yb0)
            {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                {
                    top[1][i] = bot[0][i];
                }
            }
            else
            {
                unpack(w2, top[1]);
            }
            unpack(w3, bot[1]);
        }
    }
    else
    {
        auto fetch = [&](int y, uint32_t (&t)[4])
        {
            if (y == p.srcH - 1)
            {
                fetchLast(y, t);
            }
            else
            {
                unpack(window(y), t);
            }
        };
        fetch(ya0, top[0]);
        fetch(yb0, bot[0]);
        fetch(ya1, top[1]);
        fetch(yb1, bot[1]);
    }
    pxA[0] = BilinearU8<C>(top[0][0], top[0][1], bot[0][0], bot[0][1], colA.w[0], row0.w[0]);
    pxB[0] = BilinearU8<C>(top[0][2], top[0][3], bot[0][2], bot[0][3], colB.w[0], row0.w[0]);
    pxA[1] = BilinearU8<C>(top[1][0], top[1][1], bot[1][0], bot[1][1], colA.w[0], row1.w[0]);
    pxB[1] = BilinearU8<C>(top[1][2], top[1][3], bot[1][2], bot[1][3], colB.w[0], row1.w[0]);
    // even lanes keep their first-row pair and take the neighbour's, odd lanes the same for the second row
    const uint32_t got0 = FromLaneXor1(odd ? pxA[0] : pxA[1]), got1 = FromLaneXor1(odd ? pxB[0] : pxB[1]);
    const uint32_t q[1][4] = {{odd ? got0 : pxA[0], odd ? got1 : pxB[0], odd ? pxA[1] : got0, odd ? pxB[1] : got1}};
    const int      dy = y0 + (lane & 1), dx0 = x0 + 2 * (lane & ~1);
    if (dy >= p.dstH || dx0 >= p.dstW)
    {
        return;
    }
    uint8_t *to = p.dst + (int64_t)dy * p.dstRow + (int64_t)dx0 * C;
    if (dx0 + 4 <= p.dstW)
    {
        uint32_t w[C];
        PackQuad<C>(q, w);
        StoreDwordsNT<C>(to, w);
    }
    else
    {
#pragma unroll
        for (int k = 0; k < 3; ++k)
        {
            if (dx0 + k < p.dstW)
            {
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    to[C * k + c] = (uint8_t)(q[0][k] >> (8 * c));
                }
            }
        }
    }
}

// Enlargements by 1.5 or more (3 * srcW <= 2 * dstW): the taps of FOUR neighbouring output columns lie within 4
// source pixels, so a lane owns 4 columns x 2 rows on the same window loads as the two-column form: half the loads,
// column-independent work (row terms, addresses, funnel shifts) spread over twice the pixels, and a lane's 4 pixels
// of a row are consecutive, so nothing changes lanes before the store. A wave covers 256 columns x 2 rows. The
// distance between the first and the last of a lane's four source columns is at most 2 by the scale; should
// float32 rounding ever make it 3, or the image's last row be involved, the wave takes the two-column form.
template<int C>
__device__ __forceinline__ void ResizeLinearQuadsU8(const Plane &p, int x0, int y0)
{
    if (x0 >= p.dstW || y0 >= p.dstH)
    {
        return;
    }
    const int            lane = threadIdx.x & 63;
    const int            dx0  = x0 + 4 * lane;
    AxisTerms<1>         col[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        col[j] = Axis<NVCV_INTERP_LINEAR>(p.scaleX, min(dx0 + j, p.dstW - 1), p.srcW);
    }
    const auto rows = Axis<NVCV_INTERP_LINEAR>(p.scaleY, min(y0 + (lane & 1), p.dstH - 1), p.srcH);
    const auto row0 = FromLane(rows, 0), row1 = FromLane(rows, 1);
    const int  ya0 = row0.s, yb0 = min(row0.s + 1, p.srcH - 1), ya1 = row1.s, yb1 = min(row1.s + 1, p.srcH - 1);
    const bool narrow = col[3].s - col[0].s <= 2;
    if (max(yb0, yb1) >= p.srcH - 1 || __builtin_amdgcn_ballot_w64(!narrow) != 0) // wave-uniform
    {
        ResizeLinearPairsU8<C, false>(p, x0, y0);
        ResizeLinearPairsU8<C, false>(p, x0 + 128, y0);
        return;
    }
    // pixels (s, s + 1) of column j out of the window's four
    auto taps = [&](const TapWindow<C> &win, uint32_t (&first)[4], uint32_t (&second)[4])
    {
        const uint32_t k0 = WindowPixel<C>(win, 0), k1 = WindowPixel<C>(win, 1), k2 = WindowPixel<C>(win, 2),
                       k3 = WindowPixel<C>(win, 3);
        first[0]  = k0;
        second[0] = k1;
#pragma unroll
        for (int j = 1; j < 4; ++j)
        {
            const int d = col[j].s - col[0].s;
            first[j]    = d == 0 ? k0 : (d == 1 ? k1 : k2);
            second[j]   = d == 0 ? k1 : (d == 1 ? k2 : k3);
        }
    };
    uint32_t topA[2][4], topB[2][4], botA[2][4], botB[2][4]; // [output row][column]: first and second tap, upper and lower source row
    taps(LoadTapWindow<C>(p, ya0, col[0].s), topA[0], topB[0]);
    taps(LoadTapWindow<C>(p, yb0, col[0].s), botA[0], botB[0]);
    if (ya1 == ya0)
    {
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            topA[1][j] = topA[0][j];
            topB[1][j] = topB[0][j];
            botA[1][j] = botA[0][j];
            botB[1][j] = botB[0][j];
        }
    }
    else if (ya1 == yb0)
    {
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            topA[1][j] = botA[0][j];
            topB[1][j] = botB[0][j];
        }
        taps(LoadTapWindow<C>(p, yb1, col[0].s), botA[1], botB[1]);
    }
    else
    {
        taps(LoadTapWindow<C>(p, ya1, col[0].s), topA[1], topB[1]);
        taps(LoadTapWindow<C>(p, yb1, col[0].s), botA[1], botB[1]);
    }
    if (dx0 >= p.dstW)
    {
        return;
    }
#pragma unroll
    for (int r = 0; r < 2; ++r)
    {
        const int dy = y0 + r;
        if (dy >= p.dstH)
        {
            break;
        }
        const float    wy = r == 0 ? row0.w[0] : row1.w[0];
        uint32_t       q[1][4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            q[0][j] = BilinearU8<C>(topA[r][j], topB[r][j], botA[r][j], botB[r][j], col[j].w[0], wy);
        }
        uint8_t *to = p.dst + (int64_t)dy * p.dstRow + (int64_t)dx0 * C;
        if (dx0 + 4 <= p.dstW)
        {
            uint32_t w[C];
            PackQuad<C>(q, w);
            StoreDwordsNT<C>(to, w);
        }
        else
        {
#pragma unroll
            for (int k = 0; k < 3; ++k)
            {
                if (dx0 + k < p.dstW)
                {
#pragma unroll
                    for (int c = 0; c < C; ++c)
                    {
                        to[C * k + c] = (uint8_t)(q[0][k] >> (8 * c));
                    }
                }
            }
        }
    }
}

// The windows of rows 0 .. last (wave-uniform, under 9) from `at` on, a lane's own column offset included, all of them
// requested before the first is touched: taken into place inside a test on `last`, each load would be waited for
// before the next goes out (nine round trips one after the other: 62 us instead of 51 for the two-column strips).
// The empty statement uses every raw window, so the loads can neither sink below it nor the funnel shifts rise
// above it. That all windows are in before a strip's row loop starts also keeps waits for them out of the loop:
// stores and loads share one counter of outstanding operations here, and such a wait, after rows have been stored,
// would be a wait for those stores to reach memory as well.
// 1 and 3 channels request only the windows that are needed. With 4-byte pixels the compiler joins a window that exists
// on one side of the test only to the statement through a register move, which waits for its load, so those request
// all W (rows past `last` repeat it: an L1 hit, but a load instruction; 16 x 720p -> 900p u8x3 36.8 us against
// 31.3). Two whole variants, 5 windows or 9, were slower for every pixel size (65 us for the two-column strips).
template<int C, int W>
__device__ __forceinline__ void RequestStripWindows(const uint8_t *at, int rowStride, int last, TapWindow<C> (&win)[W])
{
    RawTapWindow<C> raw[W];
#pragma unroll
    for (int k = 0; k < W; ++k)
    {
        if constexpr (C == 4)
        {
            raw[k] = RequestTapWindow<C>(at + (int64_t)min(k, last) * rowStride);
        }
        else
        {
            if (k <= last)
            {
                raw[k] = RequestTapWindow<C>(at + (int64_t)k * rowStride);
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (W == 9)
    {
        asm volatile("" ::"v"(raw[0].d[0]), "v"(raw[1].d[0]), "v"(raw[2].d[0]), "v"(raw[3].d[0]), "v"(raw[4].d[0]),
                     "v"(raw[5].d[0]), "v"(raw[6].d[0]), "v"(raw[7].d[0]), "v"(raw[8].d[0]));
    }
    else if constexpr (W == 5)
    {
        asm volatile("" ::"v"(raw[0].d[0]), "v"(raw[1].d[0]), "v"(raw[2].d[0]), "v"(raw[3].d[0]), "v"(raw[4].d[0]));
    }
    else
    {
        static_assert(W == 3);
        asm volatile("" ::"v"(raw[0].d[0]), "v"(raw[1].d[0]), "v"(raw[2].d[0]));
    }
#pragma unroll
    for (int k = 0; k < W; ++k)
    {
        win[k] = FinishTapWindow<C>(raw[k]);
    }
}

// The four-column form over a strip of R output rows per wave (kStripRows; fewer in small launches). When not reducing
// vertically those rows lie between at most R + 1 consecutive source rows. All their windows are requested up front, a source
// row's tap pairs are formed once for every output row that uses it as
// its upper or its lower row, and the column terms are paid once per R rows instead of once per 2. The blend per
// output pixel is BilinearQ15 as everywhere. A wave that reaches the image's last source row, reduces vertically
// (more source rows than fit) or has a lane whose columns do not fit its window runs as two-row steps.
constexpr int kStripRows = 8, kStripWindows = kStripRows + 1;
static_assert(kStripWindows == 9);

template<int C, int R = kStripRows>
__device__ __forceinline__ void ResizeLinearQuadStripU8(const Plane &p, int x0, int y0)
{
    constexpr int kWindows = R + 1;
    if (x0 >= p.dstW || y0 >= p.dstH)
    {
        return;
    }
    const int    lane = threadIdx.x & 63;
    const int    dx0  = x0 + 4 * lane;
    AxisTerms<1> col[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        col[j] = Axis<NVCV_INTERP_LINEAR>(p.scaleX, min(dx0 + j, p.dstW - 1), p.srcW);
    }
    // lane r holds the terms of output row y0 + r
    const auto     rows   = Axis<NVCV_INTERP_LINEAR>(p.scaleY, min(y0 + (lane & (R - 1)), p.dstH - 1), p.srcH);
    const uint32_t ayLane = FractionQ15(rows.w[0]);
    const int      yFirst = __builtin_amdgcn_readlane(rows.s, 0), yLast = __builtin_amdgcn_readlane(rows.s, R - 1) + 1;
    const bool     narrow = col[3].s - col[0].s <= 2;
    if (yLast >= p.srcH - 1 || yLast - yFirst >= kWindows || __builtin_amdgcn_ballot_w64(!narrow) != 0) // wave-uniform
    {
#pragma unroll 1
        for (int k = 0; k < R; k += 2)
        {
            ResizeLinearQuadsU8<C>(p, x0, y0 + k);
        }
        return;
    }
    TapWindow<C>   win[kWindows];
    const uint8_t *at = p.src + (int64_t)yFirst * p.srcRow + col[0].s * C;
    RequestStripWindows<C>(at, p.srcRow, yLast - yFirst, win);
    // lanes past the last column stay (the row terms are read from lanes 0 .. 7 below); they store nothing
    uint32_t ax[4];
    int      d[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        ax[j] = FractionQ15(col[j].w[0]);
        d[j]  = col[j].s - col[0].s;
    }
    // (first tap | second tap << 16) of every column and channel of a source row.
    // 1 and 3 channels: the window's four values of a channel are gathered into one dword first (two byte permutes
    // with constant selectors; for one channel the window is that dword), and a column's pair is then ONE permute
    // whose selector the lane holds (bytes d and d + 1): 18 instructions per source row where choosing the column's
    // two pixels with selects and then the channel took 27.
    uint32_t pick[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        pick[j] = 0x0c010c00u + (uint32_t)d[j] * 0x00010001u;
    }
    auto pairs = [&](const TapWindow<C> &w, uint32_t (&t)[4][C])
    {
        if constexpr (C == 4)
        {
            const uint32_t k0 = WindowPixel<C>(w, 0), k1 = WindowPixel<C>(w, 1), k2 = WindowPixel<C>(w, 2), k3 = WindowPixel<C>(w, 3);
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                const uint32_t first  = j == 0 ? k0 : (d[j] == 0 ? k0 : (d[j] == 1 ? k1 : k2));
                const uint32_t second = j == 0 ? k1 : (d[j] == 0 ? k1 : (d[j] == 1 ? k2 : k3));
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    t[j][c] = ChannelPair(first, second, c);
                }
            }
        }
        else
        {
            uint32_t x[C]; // byte k: channel c of the window's pixel k
            if constexpr (C == 1)
            {
                x[0] = w.w[0];
            }
            else
            {
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    // bytes c, c + 3, c + 6, c + 9 of the window's 12: the first two (three) lie in its first 8
                    const uint32_t third = c + 6 < 8 ? (uint32_t)(c + 6) : 0x0cu;
                    const uint32_t head  = __builtin_amdgcn_perm(w.w[1], w.w[0], (uint32_t)c | (uint32_t)(c + 3) << 8 | third << 16 | 0x0c000000u);
                    x[c] = __builtin_amdgcn_perm(w.w[2], head, 0x0100u | (c + 6 < 8 ? 2u : (uint32_t)(c + 6 - 8 + 4)) << 16 | (uint32_t)(c + 9 - 8 + 4) << 24);
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    t[j][c] = __builtin_amdgcn_perm(x[c], x[c], j == 0 ? 0x0c010c00u : pick[j]);
                }
            }
        }
    };
    const int nRows = min(R, p.dstH - y0);
    int       r     = 0;
    uint8_t  *to    = p.dst + (int64_t)y0 * p.dstRow + (int64_t)dx0 * C;
    uint32_t  top[4][C], bot[4][C];
    pairs(win[0], bot);
#pragma unroll
    for (int k = 0; k + 1 < kWindows; ++k)
    {
        if (r < nRows) // wave-uniform
        {
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    top[j][c] = bot[j][c];
                }
            }
            pairs(win[k + 1], bot);
            // the output rows between source rows yFirst + k and the next one
            while (r < nRows && __builtin_amdgcn_readlane(rows.s, r) == yFirst + k)
            {
                const uint32_t ay = __builtin_amdgcn_readlane(ayLane, r);
                uint32_t       w[C] = {}; // the row's 4 pixels as stored: every channel is rounded into its byte
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    uint32_t wt, wb;
                    WeightPairsQ15(ax[j], ay, wt, wb);
#pragma unroll
                    for (int c = 0; c < C; ++c)
                    {
                        const int at     = j * C + c;
                        w[at >> 2] = BlendQ15(top[j][c], bot[j][c], wt, wb, at & 3, w[at >> 2]);
                    }
                }
                if (dx0 + 4 <= p.dstW)
                {
                    StoreDwordsNT<C>(to, w);
                }
                else
                {
#pragma unroll
                    for (int i = 0; i < 3 * C; ++i)
                    {
                        if (dx0 + i / C < p.dstW)
                        {
                            to[i] = (uint8_t)(w[i >> 2] >> (8 * (i & 3)));
                        }
                    }
                }
                to += p.dstRow;
                ++r;
            }
        }
    }
}

// Nearest neighbour when enlarging, in the shape of the four-column strips:
// the source pixels of four neighbouring output columns lie within 4 source pixels, so a lane owns 4 columns x R
// rows, takes them from one window per source row and stores every output row that maps to that source row from
// the same registers. The wave patches spend one 3-byte load per output pixel there (8 x 720p -> 1080p u8x3: 19.0 us,
// the bilinear strips 22.9; as strips 13.6). Indices are those of Axis<NEAREST>; waves that reach the image's last row,
// reduce vertically or have a lane whose columns do not fit its window run as wave patches.
template<int C, int R>
__device__ __forceinline__ void ResizeNearestQuadStripU8(const Plane &p, int x0, int y0)
{
    if (x0 >= p.dstW || y0 >= p.dstH)
    {
        return;
    }
    const int lane = threadIdx.x & 63;
    const int dx0  = x0 + 4 * lane;
    int       s[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        s[j] = Axis<NVCV_INTERP_NEAREST>(p.scaleX, min(dx0 + j, p.dstW - 1), p.srcW).s;
    }
    // lane r holds the source row of output row y0 + r
    const int  rowLane = Axis<NVCV_INTERP_NEAREST>(p.scaleY, min(y0 + (lane & (R - 1)), p.dstH - 1), p.srcH).s;
    const int  yFirst = __builtin_amdgcn_readlane(rowLane, 0), yLast = __builtin_amdgcn_readlane(rowLane, R - 1);
    const bool narrow = s[3] - s[0] <= 3;
    if (yLast >= p.srcH - 1 || yLast - yFirst >= (R + 1) || __builtin_amdgcn_ballot_w64(!narrow) != 0) // wave-uniform
    {
#pragma unroll 1
        for (int i = 0; i < R; ++i)
        {
            ResizeWavePatch<uint8_t, C, NVCV_INTERP_NEAREST, false>(p, x0 + 64 * (i & 3), y0 + 4 * (i >> 2));
        }
        return;
    }
    TapWindow<C>   win[(R + 1)];
    const uint8_t *at = p.src + (int64_t)yFirst * p.srcRow + s[0] * C;
    RequestStripWindows<C>(at, p.srcRow, yLast - yFirst, win);
    const int nRows = min(R, p.dstH - y0);
    int       r     = 0;
    uint8_t  *to    = p.dst + (int64_t)y0 * p.dstRow + (int64_t)dx0 * C;
#pragma unroll
    for (int k = 0; k < (R + 1); ++k)
    {
        if (r < nRows) // wave-uniform
        {
            // the lane's 4 pixels of source row yFirst + k, packed as they are stored
            const uint32_t mask  = C == 4 ? 0xffffffffu : (1u << (8 * C)) - 1u;
            const uint32_t k0 = WindowPixel<C>(win[k], 0) & mask, k1 = WindowPixel<C>(win[k], 1) & mask,
                           k2 = WindowPixel<C>(win[k], 2) & mask, k3 = WindowPixel<C>(win[k], 3) & mask;
            uint32_t       q[1][4];
            q[0][0] = k0;
#pragma unroll
            for (int j = 1; j < 4; ++j)
            {
                const int d = s[j] - s[0];
                q[0][j]     = d == 0 ? k0 : (d == 1 ? k1 : (d == 2 ? k2 : k3));
            }
            uint32_t w[C];
            PackQuad<C>(q, w);
            while (r < nRows && __builtin_amdgcn_readlane(rowLane, r) == yFirst + k)
            {
                if (dx0 + 4 <= p.dstW)
                {
                    StoreDwordsNT<C>(to, w);
                }
                else
                {
#pragma unroll
                    for (int i = 0; i < 3 * C; ++i)
                    {
                        if (dx0 + i / C < p.dstW)
                        {
                            to[i] = (uint8_t)(w[i >> 2] >> (8 * (i & 3)));
                        }
                    }
                }
                to += p.dstRow;
                ++r;
            }
        }
    }
}

// Nearest neighbour of 1 and 3 channels where the output rows' source rows are not consecutive: a lane owns 4 columns as in
// the strips, but each of its R rows comes from a window of its own, DWORDS dwords from the one of the lane's first source
// pixel on. Bound by the writes: the wave patches' rows of 64 pixels (64 bytes of one channel, mostly not at a sector's start) end in
// partly written sectors twice for each, these rows of 256 once for four, and four pixels are one load instead of four. One
// channel, with inputs out of the memory's cache: 24 x 1300 x 1300 -> 1000 x 1000 26.9 -> 14.1 us, 12 x 1800 x 1800 -> 900 x 900 14.1 -> 10.2, 4 x 3000 x 3000 -> 1000 x 1000 7.9 ->
// 7.3 (in it 22.5 -> 9.8, 11.3 -> 6.3, 5.4 -> 4.8); 200 x 258 x 752 -> 244 x 711 36.7 -> 19.0. Three channels enlarged across alone (117 x 453 x 113 -> 455 x 84) 12.0 -> 10.3.
constexpr int kNearestRows = 4;

template<int C, int DWORDS>
__device__ __forceinline__ void ResizeNearestRowsU8(const Plane &p, int x0, int y0)
{
    static_assert(C == 1 ? DWORDS == 2 || DWORDS == 4 : C == 3 && DWORDS == 4);
    constexpr int R = kNearestRows;
    if (x0 >= p.dstW || y0 >= p.dstH)
    {
        return;
    }
    const int lane = threadIdx.x & 63, dx0 = x0 + 4 * lane;
    int       s[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        s[j] = Axis<NVCV_INTERP_NEAREST>(p.scaleX, min(dx0 + j, p.dstW - 1), p.srcW).s;
    }
    // lane r holds the source row of output row y0 + r
    const int  rowLane = Axis<NVCV_INTERP_NEAREST>(p.scaleY, min(y0 + (lane & (R - 1)), p.dstH - 1), p.srcH).s;
    const bool fits    = (s[3] - s[0] + 1) * C <= 4 * DWORDS - 3; // wherever in a dword the first byte is
    // (a window may run past its row, so the image's last row is left to the patches)
    if (__builtin_amdgcn_readlane(rowLane, R - 1) >= p.srcH - 1 || __builtin_amdgcn_ballot_w64(!fits) != 0) // wave-uniform
    {
#pragma unroll 1
        for (int i = 0; i < 4; ++i)
        {
            ResizeWavePatch<uint8_t, C, NVCV_INTERP_NEAREST, false>(p, x0 + 64 * i, y0);
        }
        return;
    }
    struct alignas(4) Window
    {
        uint32_t d[DWORDS];
    };
    Window   w[R];
    uint32_t at[R]; // of the first byte, from a dword in front of it on (the low two bits: in its dword)
#pragma unroll
    for (int r = 0; r < R; ++r)
    {
        const uint8_t *row = p.src + (int64_t)__builtin_amdgcn_readlane(rowLane, r) * p.srcRow;
        const uint32_t odd = (uint32_t)reinterpret_cast<uintptr_t>(row) & 3u;
        at[r]              = odd + (uint32_t)(s[0] * C);
        w[r]               = *reinterpret_cast<const Window *>(row - odd + (at[r] & ~3u));
    }
    __builtin_amdgcn_sched_barrier(0); // (every load before the first use)
    // Selectors of v_perm_b32 that make the lane's C dwords of a row from the window's bytes, counted from the first one on: of
    // the last dword, which may need bytes behind the eighth, two halves, whose missing bytes are zeros (selector 0x0c).
    constexpr bool kHalves = DWORDS > 2;
    uint32_t       low[C] = {}, high = 0;
#pragma unroll
    for (int b = 0; b < 4 * C; ++b)
    {
        const uint32_t k    = (uint32_t)((s[b / C] - s[0]) * C + b % C);
        const bool     last = kHalves && b / 4 == C - 1;
        low[b / 4] |= (last && k >= 8 ? 0x0cu : k) << (8 * (b % 4));
        high |= last ? (k >= 8 ? k - 8 : 0x0cu) << (8 * (b % 4)) : 0u;
    }
    uint8_t  *to    = p.dst + (int64_t)y0 * p.dstRow + (int64_t)dx0 * C;
    const int nRows = min(R, p.dstH - y0);
#pragma unroll
    for (int r = 0; r < R; ++r)
    {
        if (r >= nRows) // uniform
        {
            break;
        }
        uint32_t out[C];
        if constexpr (!kHalves)
        {
            out[0] = __builtin_amdgcn_perm(w[r].d[1], w[r].d[0], low[0] + (at[r] & 3u) * 0x01010101u);
        }
        else
        {
            uint32_t t[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                t[i] = __builtin_amdgcn_alignbyte(i < 3 ? w[r].d[i + 1] : 0u, w[r].d[i], at[r]);
            }
#pragma unroll
            for (int i = 0; i < C; ++i)
            {
                out[i] = __builtin_amdgcn_perm(t[1], t[0], low[i]);
            }
            out[C - 1] |= __builtin_amdgcn_perm(t[3], t[2], high);
        }
        if (dx0 + 4 <= p.dstW)
        {
            StoreDwordsNT<C>(to, out);
        }
        else
        {
#pragma unroll
            for (int i = 0; i < 3 * C; ++i)
            {
                if (dx0 + i / C < p.dstW)
                {
                    to[i] = (uint8_t)(out[i >> 2] >> (8 * (i & 3)));
                }
            }
        }
        to += p.dstRow;
    }
}

// The two-column form over strips of R output rows per wave (128 columns x 4 rows; x 2 in small launches). At vertical
// scales up to 2 those rows lie between at most 2 R + 1 consecutive source rows: the windows are requested up front, a source row
// is taken apart into its (first tap | second tap) pairs once for every output row that uses it as its upper or its
// lower row, and the column terms are paid once for all of them. Every output row is finished on its
// own: a lane rounds the channels of its 2 pixels straight into the bytes they have in the row, the lanes of a pair
// swap them, and the even lane stores the 4 pixels as whole dwords. The blend per output pixel is BilinearQ15 as
// everywhere. A wave that reaches the image's last source row or reduces vertically by more than 2 runs as
// two-row steps.
constexpr int kPairStripRows = 4;

template<int C, int R = kPairStripRows>
__device__ __forceinline__ void ResizeLinearPairStripU8(const Plane &p, int x0, int y0)
{
    constexpr int kPairStripWindows = 2 * R + 1;
    if (x0 >= p.dstW || y0 >= p.dstH)
    {
        return;
    }
    const int lane = threadIdx.x & 63;
    const int dx0  = x0 + 2 * lane;
    // columns and rows past the output compute a duplicate of the last one: every lane takes part in the swap
    const auto colA  = Axis<NVCV_INTERP_LINEAR>(p.scaleX, min(dx0, p.dstW - 1), p.srcW);
    const auto colB  = Axis<NVCV_INTERP_LINEAR>(p.scaleX, min(dx0 + 1, p.dstW - 1), p.srcW);
    const int  delta = colB.s - colA.s; // 0 .. 2 at scales up to 2
    // lane r holds the terms of output row y0 + r
    const auto     rows   = Axis<NVCV_INTERP_LINEAR>(p.scaleY, min(y0 + (lane & (R - 1)), p.dstH - 1), p.srcH);
    const uint32_t ayLane = FractionQ15(rows.w[0]);
    const int      yFirst = __builtin_amdgcn_readlane(rows.s, 0), yLast = __builtin_amdgcn_readlane(rows.s, R - 1) + 1;
    if (yLast >= p.srcH - 1 || yLast - yFirst >= kPairStripWindows) // wave-uniform
    {
#pragma unroll
        for (int r = 0; r < R; r += 2)
        {
            ResizeLinearPairsU8<C, false>(p, x0, y0 + r);
        }
        return;
    }
    TapWindow<C>   win[kPairStripWindows];
    const uint8_t *at = p.src + (int64_t)yFirst * p.srcRow + colA.s * C;
    RequestStripWindows<C>(at, p.srcRow, yLast - yFirst, win);
    const uint32_t axA = FractionQ15(colA.w[0]), axB = FractionQ15(colB.w[0]);
    // (first tap | second tap << 16) of both columns and every channel of a source row
    auto pairs = [&](const TapWindow<C> &w, uint32_t (&t)[2][C])
    {
        const uint32_t k0 = WindowPixel<C>(w, 0), k1 = WindowPixel<C>(w, 1), k2 = WindowPixel<C>(w, 2), k3 = WindowPixel<C>(w, 3);
        const uint32_t first = delta == 0 ? k0 : (delta == 1 ? k1 : k2), second = delta == 0 ? k1 : (delta == 1 ? k2 : k3);
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            t[0][c] = ChannelPair(k0, k1, c);
            t[1][c] = ChannelPair(first, second, c);
        }
    };
    const int  nRows = min(R, p.dstH - y0);
    const bool even  = (lane & 1) == 0;
    int        r     = 0;
    uint8_t   *to    = p.dst + (int64_t)y0 * p.dstRow + (int64_t)dx0 * C; // (used by even lanes: 4 pixels from their first)
    uint32_t   top[2][C], bot[2][C];
    pairs(win[0], bot);
#pragma unroll
    for (int k = 0; k + 1 < kPairStripWindows; ++k)
    {
        if (r < nRows) // wave-uniform
        {
#pragma unroll
            for (int j = 0; j < 2; ++j)
            {
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    top[j][c] = bot[j][c];
                }
            }
            pairs(win[k + 1], bot);
            // the output rows between source rows yFirst + k and the next one
            while (r < nRows && __builtin_amdgcn_readlane(rows.s, r) == yFirst + k)
            {
                const uint32_t ay = __builtin_amdgcn_readlane(ayLane, r);
                // the lane's 2 pixels as the 2 C bytes they are in the row
                uint32_t mine[2] = {0, 0};
#pragma unroll
                for (int j = 0; j < 2; ++j)
                {
                    uint32_t wt, wb;
                    WeightPairsQ15(j == 0 ? axA : axB, ay, wt, wb);
#pragma unroll
                    for (int c = 0; c < C; ++c)
                    {
                        const int at8 = j * C + c;
                        mine[at8 >> 2] = BlendQ15(top[j][c], bot[j][c], wt, wb, at8 & 3, mine[at8 >> 2]);
                    }
                }
                // the even lane takes its neighbour's and stores 4 pixels
                uint32_t w[C];
                if constexpr (C == 4)
                {
                    w[0] = mine[0];
                    w[1] = mine[1];
                    w[2] = FromLaneXor1(mine[0]);
                    w[3] = FromLaneXor1(mine[1]);
                }
                else if constexpr (C == 3)
                {
                    const uint32_t lo = FromLaneXor1(mine[0]), hi = FromLaneXor1(mine[1]);
                    w[0] = mine[0];
                    w[1] = mine[1] | (lo << 16);
                    w[2] = __builtin_amdgcn_alignbit(hi, lo, 16);
                }
                else
                {
                    static_assert(C == 1);
                    w[0] = mine[0] | (FromLaneXor1(mine[0]) << 16);
                }
                if (even && dx0 < p.dstW)
                {
                    if (dx0 + 4 <= p.dstW)
                    {
                        StoreDwordsNT<C>(to, w);
                    }
                    else
                    {
#pragma unroll
                        for (int i = 0; i < 3 * C; ++i)
                        {
                            if (dx0 + i / C < p.dstW)
                            {
                                to[i] = (uint8_t)(w[i >> 2] >> (8 * (i & 3)));
                            }
                        }
                    }
                }
                to += p.dstRow;
                ++r;
            }
        }
    }
}

// Which (type, channels, interpolation) take the two-columns-per-lane form. The code is written for 1, 3
// and 4 channels; with 1 and 4 it measured slower than the wave patches (u8x1 43 -> 58 us, u8x4 91 -> 104 us
// on 1080p -> 720p: the column terms of two columns are amortised over 2 rows only), so 3 it is.
template<class T, int C, int INTERP>
constexpr bool kPairsForm = std::is_same_v<T, uint8_t> && INTERP == NVCV_INTERP_LINEAR && (C == 1 || C == 3 || C == 4);

// The scales at which the two-column form is the faster one (per image): horizontal scales up to 2; 4-byte pixels
// only when not reducing (16 x 1080p -> 720p: 34.4 us against the wave patches' 29.9; 720p -> 900p: 37.9 against 42.0).
template<int C>
__host__ __device__ __forceinline__ bool PairsFormScale(int srcW, int dstW)
{
    return srcW >= 4 && srcW <= 2 * dstW && (C != 4 || srcW <= dstW);
}

constexpr int kPairsTileW = 128, kPairsTileH = 8; // image batches: block = 4 waves of 128 columns x 2 rows, stacked

template<int C, int R>
__global__ __launch_bounds__(256) void ResizeLinearPairsU8Kernel(const ResizeArgs a, const WaveOrder order)
{
    const Plane p = GetPlanes<false>(a, blockIdx.z);
    const WaveTile t = WaveTileOf(order);
    ResizeLinearPairStripU8<C, R>(p, t.x * kPairsTileW, t.y * R);
}

constexpr int kQuadsTileW = 256; // a wave's columns; where a block's waves stand: WaveTileOf

template<int C, int R>
__global__ __launch_bounds__(256) void ResizeLinearQuadsU8Kernel(const ResizeArgs a, const WaveOrder order)
{
    const Plane p = GetPlanes<false>(a, blockIdx.z);
    const WaveTile t = WaveTileOf(order);
    ResizeLinearQuadStripU8<C, R>(p, t.x * kQuadsTileW, t.y * R);
}

template<int C, int R>
__global__ __launch_bounds__(256) void ResizeNearestQuadsU8Kernel(const ResizeArgs a, const WaveOrder order)
{
    const Plane p = GetPlanes<false>(a, blockIdx.z);
    const WaveTile t = WaveTileOf(order);
    ResizeNearestQuadStripU8<C, R>(p, t.x * kQuadsTileW, t.y * R);
}

template<int C, int DWORDS>
__global__ __launch_bounds__(256) void ResizeNearestRowsU8Kernel(const ResizeArgs a, const WaveOrder order)
{
    const Plane p = GetPlanes<false>(a, blockIdx.z);
    const WaveTile t = WaveTileOf(order);
    ResizeNearestRowsU8<C, DWORDS>(p, t.x * kQuadsTileW, t.y * kNearestRows);
}

// Image batches: the same 128 x 8 tile per block for every image; an image whose horizontal scale is
// above 2 (or whose source is narrower than 4 pixels) is resized as four 64 x 4 wave patches instead.
template<int C>
__global__ __launch_bounds__(256) void ResizeLinearPairsU8VarShapeKernel(const ResizeArgs a, const VarTiles tiles)
{
    const TileCoord tc   = LocateTile(tiles, blockIdx.x);
    const Plane     p    = GetPlanes<true>(a, tc.image);
    const int       wave = threadIdx.x >> 6;
    if (PairsFormScale<C>(p.srcW, p.dstW))
    {
        ResizeLinearPairsU8<C, true>(p, tc.tx * kPairsTileW, tc.ty * kPairsTileH + wave * 2);
    }
    else
    {
        ResizeWavePatch<uint8_t, C, NVCV_INTERP_LINEAR, true>(p, tc.tx * kPairsTileW + (wave & 1) * 64,
                                                             tc.ty * kPairsTileH + (wave >> 1) * 4);
    }
}

// Large image-batch launches resize each image in the tensor kernels' strips; a wave owns a tile of 256 x 8 (WIDE: most of
// the launch is enlarged by 1.5 or more) or 128 x 4 output pixels, a block four of them, side by side or stacked
// (VarWaveTileOf; the host chooses by the images' widths). WIDE: four columns per lane where the
// image is enlarged so, else two columns per lane at horizontal scales up to 2 (4 strips of 128 x 4), else 8 wave
// patches. Otherwise a two-column strip, or two wave patches.
template<bool WIDE>
constexpr int kStripsWaveW = WIDE ? kQuadsTileW : kPairsTileW;
template<bool WIDE>
constexpr int kStripsWaveH = WIDE ? kStripRows : kPairStripRows;

// The tile (in units of a wave's tile) of this wave in an image-batch block whose tile is 4 wave tiles wide (flat) or high.
__device__ __forceinline__ WaveTile VarWaveTileOf(const TileCoord &tc, int flat)
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), f = flat != 0;
    return WaveTile{tc.tx * (3 * f + 1) + wave * f, tc.ty * (4 - 3 * f) + wave * (1 - f)};
}

template<int C>
__host__ __device__ __forceinline__ bool QuadStripScale(int srcW, int dstW)
{
    return srcW >= 4 && 3 * (int64_t)srcW <= 2 * (int64_t)dstW;
}

template<int C, bool WIDE>
__global__ __launch_bounds__(256) void ResizeLinearStripsU8VarShapeKernel(const ResizeArgs a, const VarTiles tiles, const int flat)
{
    const TileCoord tc = LocateTile(tiles, blockIdx.x);
    const Plane     p  = GetPlanes<true>(a, tc.image);
    const WaveTile  t  = VarWaveTileOf(tc, flat);
    const int       x0 = t.x * kStripsWaveW<WIDE>, y0 = t.y * kStripsWaveH<WIDE>;
    if constexpr (WIDE)
    {
        if (QuadStripScale<C>(p.srcW, p.dstW))
        {
            ResizeLinearQuadStripU8<C>(p, x0, y0);
        }
        else if (PairsFormScale<C>(p.srcW, p.dstW))
        {
#pragma unroll 1
            for (int i = 0; i < 4; ++i)
            {
                ResizeLinearPairStripU8<C>(p, x0 + (i & 1) * kPairsTileW, y0 + (i >> 1) * kPairStripRows);
            }
        }
        else
        {
#pragma unroll 1
            for (int i = 0; i < 8; ++i)
            {
                ResizeWavePatch<uint8_t, C, NVCV_INTERP_LINEAR, true>(p, x0 + (i & 3) * 64, y0 + (i >> 2) * 4);
            }
        }
    }
    else
    {
        if (PairsFormScale<C>(p.srcW, p.dstW))
        {
            ResizeLinearPairStripU8<C>(p, x0, y0);
        }
        else
        {
            ResizeWavePatch<uint8_t, C, NVCV_INTERP_LINEAR, true>(p, x0, y0);
            ResizeWavePatch<uint8_t, C, NVCV_INTERP_LINEAR, true>(p, x0 + 64, y0);
        }
    }
}

// Nearest neighbour: whether an image takes the four-column strips (enlarged by 1.5 or more across, not reduced down;
// a window may start at a row's last pixel and, with the bytes a load takes along, runs up to 13
// bytes into the next row: sources of 8 columns and more).
template<int C>
__host__ __device__ __forceinline__ bool NearestStripScale(int srcW, int srcH, int dstW, int dstH)
{
    return srcW >= 8 && 3 * (int64_t)srcW <= 2 * (int64_t)dstW && srcH <= dstH;
}

// Image batches that are mostly such images: a 256 x R tile per wave (4 or 8 rows), a strip or patches.
template<int C, int R>
__global__ __launch_bounds__(256) void ResizeNearestStripsU8VarShapeKernel(const ResizeArgs a, const VarTiles tiles, const int flat)
{
    const TileCoord tc = LocateTile(tiles, blockIdx.x);
    const Plane     p  = GetPlanes<true>(a, tc.image);
    const WaveTile  t  = VarWaveTileOf(tc, flat);
    const int       x0 = t.x * kStripsWaveW<true>, y0 = t.y * R;
    if (NearestStripScale<C>(p.srcW, p.srcH, p.dstW, p.dstH))
    {
        ResizeNearestQuadStripU8<C, R>(p, x0, y0);
    }
    else
    {
#pragma unroll 1
        for (int i = 0; i < R; ++i)
        {
            ResizeWavePatch<uint8_t, C, NVCV_INTERP_NEAREST, true>(p, x0 + (i & 3) * 64, y0 + (i >> 2) * 4);
        }
    }
}

constexpr int kPatchTileW = 64, kPatchTileH = 16; // block = 4 waves stacked vertically

template<class T, int C, int INTERP, bool ODD>
__global__ __launch_bounds__(256) void ResizePatchTensorKernel(const ResizeArgs a, const WaveOrder order)
{
    const Plane p = GetPlanes<false>(a, blockIdx.z);
    // blocks are 4 waves, or single waves when the whole launch is small
    const WaveTile t = WaveTileOf(order);
    ResizeWavePatch<T, C, INTERP, false, ODD>(p, t.x * kPatchTileW, t.y * 4);
}

// ---- the 8-bit bicubic form that walks the source rows once
//
// Sizes that it takes: every source row counts (farther apart, rows between the windows would be summed for nothing), loads of
// 16 bytes (8 for one channel) fit a row, and a lane's columns fit its loads, and half of a wave's lanes
// have columns (one channel, 128 x 64 x 64 -> 48 x 48: as patches 3.6 us, so 4.7; three channels need a whole tile, see below).
template<int C>
constexpr int kCubicWalkW = C == 1 ? 256 : 64; // a wave's columns

constexpr int kCubicBatchRows = 16; // image batches: a wave's rows

template<int C>
__host__ __device__ __forceinline__ bool CubicWalks(int srcW, int srcH, int dstW, int dstH)
{
    return srcH >= 4 && srcH <= 4 * (int64_t)dstH && srcW * C >= (C == 1 ? 8 : 16)
        && dstW >= (C == 1 ? 128 : C == 3 ? 64 : 1) && (C != 1 || 10 * (int64_t)srcW <= 39 * (int64_t)dstW);
}

// What a lane knows of its columns, and its part of a source row. One channel: four columns, which lie within 8 source
// bytes (LOADS = 1, horizontal scales up to 1.3) or two by two (LOADS = 2, up to 3.9): a row is one or two unaligned 8-byte
// loads, and two byte permutes whose selectors are the column's for all rows bring its taps side by side. Windows of columns
// near the row's end start 8 bytes before it. Three and four channels: one column, its window as LoadQuadWindow reads it.
template<int C, int LOADS, bool ODD>
struct CubicLane
{
    static constexpr int K = C == 1 ? 4 : 1; // columns
    static constexpr int D = C == 1 ? 2 : 4; // dwords of a load

    struct Window
    {
        uint32_t d[LOADS][D];
        uint32_t shift; // three channels: the window's place in its dwords (the low two bits)
    };

    uint32_t at[LOADS], pick[K], w01[K], w23[K]; // pick: one channel: the permute of taps 0 and 1; else the window's byte offset

    __device__ __forceinline__ CubicLane(const Plane &p, int x)
    {
#pragma unroll
        for (int k = 0; k < K; ++k)
        {
            const auto           col = FinishedAxis<NVCV_INTERP_CUBIC>(p.scaleX, x + k, p.srcW, true);
            const CubicColumnQ14 cq  = CubicColumn<C>(col);
            w01[k]                   = cq.w01;
            w23[k]                   = cq.w23;
            if constexpr (C == 1)
            {
                const int l = k * LOADS / K;
                if (k % (K / LOADS) == 0)
                {
                    at[l] = (uint32_t)min(col.s - 1, p.srcW - 8);
                }
                pick[k] = 0x0c010c00u + ((uint32_t)(col.s - 1) - at[l]) * 0x00010001u;
            }
            else
            {
                at[0]   = cq.at;
                pick[0] = cq.at + cq.shift;
            }
        }
    }

    // Where a window of three channels begins: row `row` of the image from its own first dword of memory on, the image's last
    // row from its first byte on and ending with it at the latest.
    __device__ __forceinline__ uint32_t Begin(const Plane &p, const uint8_t *line, bool end, uint32_t &mis) const
    {
        mis              = ODD && !end ? RowMisalignment(line) : 0u;
        const uint32_t o = ODD ? (pick[0] + mis) & ~3u : at[0];
        return min(o, end ? (uint32_t)p.srcW * C - 4 * D : ~0u);
    }

    __device__ __forceinline__ Window Request(const Plane &p, int row) const
    {
        const uint8_t *line = p.src + (int64_t)min(row, p.srcH - 1) * p.srcRow;
        struct __attribute__((packed, aligned(1))) Bytes
        {
            uint32_t d[D];
        };
        Window w;
#pragma unroll
        for (int l = 0; l < LOADS; ++l)
        {
            uint32_t off = at[l], mis = 0;
            if constexpr (C == 3)
            {
                off = Begin(p, line, row >= p.srcH - 1, mis);
            }
            // (stays a 32-bit offset to a scalar base: widened ahead of the loop it takes 64-bit sums per lane)
            asm("" : "+v"(off));
            const Bytes b = *reinterpret_cast<const Bytes *>(line - mis + off);
            __builtin_memcpy(w.d[l], &b, sizeof(b));
        }
        return w;
    }

    // The same of any row but the image's last, `line`.
    __device__ __forceinline__ Window RequestInner(const uint8_t *line)
    {
        struct __attribute__((packed, aligned(1))) Bytes
        {
            uint32_t d[D];
        };
        Window   w;
        uint32_t mis = 0;
        if constexpr (ODD)
        {
            mis     = RowMisalignment(line);
            w.shift = pick[0] + mis;
        }
#pragma unroll
        for (int l = 0; l < LOADS; ++l)
        {
            uint32_t off;
            if constexpr (ODD)
            {
                off = w.shift & ~3u;
                asm("" : "+v"(off)); // (as above)
            }
            else
            {
                asm("" : "+v"(at[l])); // (in place: a copy is a move for each row)
                off = at[l];
            }
            const Bytes b = *reinterpret_cast<const Bytes *>(line - mis + off);
            __builtin_memcpy(w.d[l], &b, sizeof(b));
        }
        return w;
    }

    // The window's sums of 4 taps times the horizontal weights, C for each column (units of 2^-14). INNER: as RequestInner read it.
    template<bool INNER>
    __device__ __forceinline__ void Sums(const Plane &p, int row, const Window &w, float (&h)[K * C]) const
    {
        if constexpr (C == 1)
        {
#pragma unroll
            for (int k = 0; k < K; ++k)
            {
                const uint32_t(&d)[D] = w.d[k * LOADS / K];
                h[k] = RowSumQ14(__builtin_amdgcn_perm(d[1], d[0], pick[k]), __builtin_amdgcn_perm(d[1], d[0], pick[k] + 0x00020002u),
                                 w01[k], w23[k]);
            }
        }
        else
        {
            uint32_t r[C];
            if constexpr (C == 4)
            {
                __builtin_memcpy(r, w.d[0], sizeof(r));
            }
            else if constexpr (INNER)
            {
#pragma unroll
                for (int i = 0; i < C; ++i)
                {
                    r[i] = __builtin_amdgcn_alignbyte(w.d[0][i + 1], w.d[0][i], ODD ? w.shift : pick[0]);
                }
            }
            else
            {
                const bool     end  = row >= p.srcH - 1;
                const uint8_t *line = p.src + (int64_t)min(row, p.srcH - 1) * p.srcRow;
                uint32_t       mis;
                const uint32_t begin = Begin(p, line, end, mis), shift = pick[0] + mis - begin; // (4 only if moved back)
#pragma unroll
                for (int i = 0; i < C; ++i)
                {
                    r[i] = __builtin_amdgcn_alignbyte(w.d[0][i + 1], w.d[0][i], shift);
                }
                if (end && shift == 4)
                {
                    __builtin_memcpy(r, &w.d[0][1], sizeof(r));
                }
            }
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                h[c] = RowSumQ14(QuadTapPair<C>(r, 0, c), QuadTapPair<C>(r, 2, c), w01[0], w23[0]);
            }
        }
    }
};

// A wave owns 64 lanes' columns x `rows` output rows (64 at most). It walks down the source rows, keeps the sums of the last
// four in registers (a row's place is its number modulo 4, four steps unrolled) and finishes the output rows whose window ends
// with the row just added: every sum is formed once per strip, at any scale, and none is added with weight 0. Rows are
// requested two steps ahead (four were no faster; eight at a time, 22.7 us for 17.2: the registers). The vertical weights wait
// in LDS, one broadcast read per output row (as v_readlane 8 % slower). Sums, their order and the result are those of
// CubicRowsQ14 bit for bit.
// An output row leaves as one dword per lane; three channels: the three bytes of four lanes as three of their dwords.
template<int C, int LOADS, bool ODD>
__device__ __forceinline__ void ResizeCubicWalkU8(const Plane &p, int x0, int y0, int rows)
{
    using Lane       = CubicLane<C, LOADS, ODD>;
    constexpr int K  = Lane::K, V = K * C;
    const int     lane = threadIdx.x & 63, n = min(rows, p.dstH - y0);
    if (x0 >= p.dstW || n <= 0)
    {
        return;
    }
    if constexpr (C == 3)
    {
        x0 = min(x0, p.dstW - 64); // (the last tile overlaps its neighbour, with the same values; so do one channel's last columns)
    }
    const int  x = min(x0 + K * lane, p.dstW - K);
    Lane       column(p, x);
    const auto down = FinishedAxis<NVCV_INTERP_CUBIC>(p.scaleY, min(y0 + lane, p.dstH - 1), p.srcH, false); // lane r: output row y0 + r
    __shared__ float4 weights[4][64];
    float4           *wy    = weights[threadIdx.x >> 6];
    constexpr float   kUnit = 1.f / 16384.f; // the row sums'
    wy[lane] = make_float4(down.w[0] * kUnit, down.w[1] * kUnit, down.w[2] * kUnit, down.w[3] * kUnit);
    WaveExchangeFence();

    // three channels: lane 4 g + i, i < 3, holds dword i of the group's 12 bytes
    constexpr uint32_t kThird[4] = {0x04020100u, 0x05040201u, 0x06050402u, 0x06050402u};
    const int          part      = lane & 3;
    const uint32_t     third     = part == 0 ? kThird[0] : part == 1 ? kThird[1] : kThird[2];
    uint32_t           to        = C == 3 ? (uint32_t)(x0 + (lane & ~3)) * 3 + 4 * part : (uint32_t)x * C;
    const bool         mine      = C == 3 ? part != 3 : x0 + K * lane < p.dstW;

    auto walk = [&](auto inner)
    {
        constexpr bool kInner = decltype(inner)::value;
        int            j      = __builtin_amdgcn_readlane(down.s, 0) - 1; // the row whose sums come next
        const uint8_t *line   = p.src + (int64_t)j * p.srcRow;           // the row to be requested next, `ahead` of it
        auto           request = [&](int row)
        {
            if constexpr (kInner)
            {
                const auto w = column.RequestInner(line);
                line += p.srcRow;
                return w;
            }
            else
            {
                return column.Request(p, row);
            }
        };
        float h[4][V];
        {
            const auto r0 = request(j), r1 = request(j + 1), r2 = request(j + 2);
            column.template Sums<kInner>(p, j, r0, h[0]);
            column.template Sums<kInner>(p, j + 1, r1, h[1]);
            column.template Sums<kInner>(p, j + 2, r2, h[2]);
        }
        j += 3;
        typename Lane::Window ahead[2];
        ahead[0] = request(j);
        ahead[1] = request(j + 1);
        uint8_t *out = p.dst + (int64_t)y0 * p.dstRow;
        int      r = 0, last = j; // the output row to come, and the last row of its window
        float4   w = wy[0];
        for (;;)
        {
#pragma unroll
            for (int u = 0; u < 4; ++u, ++j)
            {
                const auto now = ahead[u & 1];
                ahead[u & 1]   = request(j + 2);
                column.template Sums<kInner>(p, j, now, h[(3 + u) & 3]);
                while (last <= j) // (equal: windows of later rows do not end earlier)
                {
                    uint32_t q = 0;
#pragma unroll
                    for (int k = 0; k < V; ++k)
                    {
                        float v = h[u & 3][k] * w.x;
                        v       = fmaf(h[(u + 1) & 3][k], w.y, v);
                        v       = fmaf(h[(u + 2) & 3][k], w.z, v);
                        v       = fmaf(h[(u + 3) & 3][k], w.w, v);
                        q       = __builtin_amdgcn_cvt_pk_u8_f32(fabsf(v), k, q);
                    }
                    if constexpr (C == 3)
                    {
                        const uint32_t next = (uint32_t)__builtin_amdgcn_mov_dpp((int)q, 0xF9 /* quad_perm 1,2,3,3 */, 0xF, 0xF, false);
                        q                   = __builtin_amdgcn_perm(next, q, third);
                    }
                    if (mine)
                    {
                        asm("" : "+v"(to)); // (as in Request)
                        StoreDwordsNT<1>(out + to, {q});
                    }
                    if (++r >= n)
                    {
                        return;
                    }
                    w = wy[r];
                    out += p.dstRow;
                    last = __builtin_amdgcn_readlane(down.s, r) + 2;
                }
            }
        }
    };
    // Rows are requested up to two behind the last one that is used. Strips clear of the image's last row need neither its test nor its
    // guarded offsets for each row, a third of a row's vector instructions (three channels, 16 x 1283 x 721 -> 1931 x 1081 52.3 -> 43.4 us, 2 x
    // 2608 x 1933 -> 4096 x 4000 42.0 -> 37.6, 32 x 720p -> 1080p 94.5 -> 90.1, 64 x 256 x 256 -> 224 x 224 9.6 -> 8.7; four up to 2 %). One channel
    // has no such offsets and pays for the second copy with registers: 32 x 720p -> 1080p 25.6 and 25.9.
    if (C != 1 && __builtin_amdgcn_readlane(down.s, n - 1) + 4 < p.srcH - 1)
    {
        walk(std::bool_constant<C != 1>{});
    }
    else
    {
        walk(std::false_type{});
    }
}

template<int C, int LOADS, bool ODD>
__global__ __launch_bounds__(256) void ResizeCubicWalkU8Kernel(const ResizeArgs a, const int rows, const WaveOrder order)
{
    const Plane    p = GetPlanes<false>(a, blockIdx.z);
    const WaveTile t = WaveTileOf(order);
    ResizeCubicWalkU8<C, LOADS, ODD>(p, t.x * kCubicWalkW<C>, t.y * rows, rows);
}

// Large image batches: a 64 x 64 tile per block, 16 rows of it per wave, walked where the image's sizes allow, else as four
// patches.
template<int C, bool ODD>
__global__ __launch_bounds__(256) void ResizeCubicWalkU8VarShapeKernel(const ResizeArgs a, const VarTiles tiles)
{
    const TileCoord tc = LocateTile(tiles, blockIdx.x);
    const Plane     p  = GetPlanes<true>(a, tc.image);
    const int       x0 = tc.tx * kPatchTileW, y0 = (tc.ty * 4 + (int)(threadIdx.x >> 6)) * kCubicBatchRows;
    if (CubicWalks<C>(p.srcW, p.srcH, p.dstW, p.dstH))
    {
        ResizeCubicWalkU8<C, 1, ODD>(p, x0, y0, kCubicBatchRows);
        return;
    }
#pragma unroll 1
    for (int g = 0; g < kCubicBatchRows; g += 4)
    {
        ResizeWavePatch<uint8_t, C, NVCV_INTERP_CUBIC, true, ODD>(p, x0, y0 + g);
    }
}

template<class T, int C, int INTERP, bool ODD>
__global__ __launch_bounds__(256) void ResizePatchVarShapeKernel(const ResizeArgs a, const VarTiles tiles, const int flat)
{
    const TileCoord tc = LocateTile(tiles, blockIdx.x);
    const Plane     p  = GetPlanes<true>(a, tc.image);
    const WaveTile  t  = VarWaveTileOf(tc, flat);
    ResizeWavePatch<T, C, INTERP, true, ODD>(p, t.x * kPatchTileW, t.y * 4);
}

// ---------------------------------------------------------------------------------------------
// Box filter (AREA) of 8-bit pixels at reductions of up to 3 along both axes, in fixed point.
//
// The weight of a source pixel is the length of its overlap with the box the output pixel covers,
// [d * scale, d * scale + scale): for scales of 1 and more exactly the reference's left-partial, whole and
// right-partial weights (cuda_tools/InterpolationWrap.hpp:668-760; each is one float32 subtraction of the
// same operands), pixels outside the image weigh nothing, and the sum is divided by the length of the box
// inside the image along each axis. A box of up to 3 touches at most 4 pixels per axis; the window of 4
// starts at the box's first pixel or, at the image's far edge, 4 before its end (pixels in front of the box
// then get the weight 0 from the same expression), so a window never leaves its row. Per source row the 4
// pixels are one load of the dwords that hold them; the horizontal weights, already divided, are rounded to
// 15 bits and a row's sum is two v_dot2_u32_u16 per channel on bytes (exact, below 2^24); the rows' sums are
// added in float32 with the rows' weights (wave-uniform), and the result is rounded once.
//
// One wave produces 64 columns x 16 rows: lane l owns column l (its terms are computed once), the 16 rows'
// terms are computed side by side in lanes 0-15 and read back as wave-uniform values, and every 4 rows leave
// through the 4x4 lane transposes as whole dwords.
template<class T, int C, int INTERP>
constexpr bool kAreaFixed = std::is_same_v<T, uint8_t> && INTERP == NVCV_INTERP_AREA && (C == 1 || C == 3 || C == 4);

constexpr int kAreaRowsMost = 16; // output rows per wave: 4, 8 or 16
constexpr int kAreaTileW = 64;    // image batches: block = 4 waves stacked vertically; tensors: along the rows (WaveTileOf)

// Rows per wave, given the launch's waves of 16. A wave's steps of 4 rows follow one another, so a launch that does not fill
// the chip takes as long as one wave: fewer steps each until there are enough of them. us with 16 / 8 / 4 rows, three
// channels: 224 x 224 -> 112 x 112 7.4 / 5.2 / 3.9; 640 x 480 -> 320 x 240 7.7 / 5.0 / 3.8; 1080p -> 720p 6.2 / 5.5 / 5.2; 32 x 256 x
// 256 -> 224 x 224 9.5 / 8.6 / 8.3; 16 x 640 x 480 -> 416 x 416 12.8 / 11.2 / 11.6; 8 x 1080p -> 720p 18.0 / 17.4 / 19.4; 16 of these
// 31.1 / 31.5 / 36.1, one channel 19.7 / 20.9 / 25.5: the column terms are paid per wave.
int AreaRowsPerWave(int64_t waves)
{
    return waves <= 8 * 256 ? 4 : waves <= 32 * 256 ? 8 : kAreaRowsMost;
}

// Per image: both scales within 1 .. 3 and a source of at least 4 rows of at least 32 bytes.
__host__ __device__ __forceinline__ bool AreaFixedDomain(float scaleX, float scaleY, int srcRowBytes, int srcH)
{
    return scaleX >= 1.f && scaleX <= 3.f && scaleY >= 1.f && scaleY <= 3.f && srcRowBytes >= 32 && srcH >= 4;
}

// Weights of the 4 source indices from `start` on (a whole number) for output index d: each one's overlap with
// the box, divided by the box's length inside the image, times `unit`. The overlap of index x is written
// clamp(f2 - x, 0, 1) - clamp(f1 - x, 0, 1) (a clamp is one v_med3_f32): for an index the box
// covers partly, wholly or not at all that is f2 - x or (x + 1) - f1 (both exact), 1, or 0. With `bounded`,
// indices behind the image weigh nothing (callers that pass a start of at most srcSize - 4 need no test).
__device__ __forceinline__ void AreaWeights(float scale, int d, int srcSize, float unit, float start, bool bounded, float (&w)[4])
{
    const float f1 = d * scale, end = f1 + scale;
    const float f2 = bounded ? fminf(end, (float)srcSize) : end;
    const float norm = (1.f / fminf(scale, srcSize - f1)) * unit;
    float       x = start;
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        w[k] = (__builtin_amdgcn_fmed3f(f2 - x, 0.f, 1.f) - __builtin_amdgcn_fmed3f(f1 - x, 0.f, 1.f)) * norm;
        x += 1.f;
    }
}

__device__ __forceinline__ uint32_t Dot2U16(uint32_t taps, uint32_t weights, uint32_t acc)
{
    typedef unsigned short U16x2 __attribute__((ext_vector_type(2)));
    U16x2 t, w;
    __builtin_memcpy(&t, &taps, 4);
    __builtin_memcpy(&w, &weights, 4);
    return __builtin_amdgcn_udot2(t, w, acc, false);
}

// A source row's sums per channel from its window and the packed horizontal weights, each plus 2^23: the integer sum
// (below 2^23) is accumulated on the bit pattern of 8388608.0f, whose unit in the last place is 1, so the register
// read as a float IS 2^23 + sum and no conversion is needed. The caller's accumulator starts at minus 2^23 times
// the sum of the rows' weights.
template<int C>
__device__ __forceinline__ void AreaRowSums(const uint32_t (&r)[C], uint32_t w01, uint32_t w23, float (&s)[C])
{
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        s[c] = __uint_as_float(Dot2U16(QuadTapPair<C>(r, 2, c), w23, Dot2U16(QuadTapPair<C>(r, 0, c), w01, 0x4b000000u)));
    }
}

// K output pixels per lane (vertically adjacent) from N source rows, the first at `row`; wy[k][j] is the weight of
// source row j in output pixel k. All N windows are requested before the first sum; every row's sums are formed once.
// Rows are added in ascending order, the first as a product, the others with fused multiply-adds: a row of weight 0
// changes nothing, so the result does not depend on which rows are passed beside those of the pixel's box.
template<int C, int N, int K>
__device__ __forceinline__ void AreaSumRows(const uint32_t (&r)[N][C], uint32_t w01, uint32_t w23, const float (&wy)[K][4],
                                            const float (&start)[K], uint32_t *out)
{
    float acc[K][C];
#pragma unroll
    for (int j = 0; j < N; ++j)
    {
        float s[C];
        AreaRowSums<C>(r[j], w01, w23, s);
#pragma unroll
        for (int k = 0; k < K; ++k)
        {
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                acc[k][c] = fmaf(s[c], wy[k][j], j == 0 ? start[k] : acc[k][c]);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < K; ++k)
    {
        out[k] = 0;
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            out[k] = __builtin_amdgcn_cvt_pk_u8_f32(acc[k][c], c, out[k]);
        }
    }
}

template<int C, int N, int K, bool GUARDED, bool ODD>
__device__ __forceinline__ void AreaFixedPixels(const uint8_t *row, int srcRow, int lastRowIn, uint32_t at, uint32_t shift,
                                                uint32_t rowBytes, uint32_t w01, uint32_t w23, const float (&wy)[K][4],
                                                const float (&start)[K], uint32_t (&out)[K])
{
    uint32_t r[N][C];
#pragma unroll
    for (int j = 0; j < N; ++j)
    {
        LoadQuadWindow<C, GUARDED, ODD>(row + (int64_t)j * srcRow, at, shift, j == lastRowIn, rowBytes, r[j]);
    }
    AreaSumRows<C, N, K>(r, w01, w23, wy, start, out);
}

// Two such pairs of output pixels (4 vertically adjacent ones) from 3 source rows each, none of them the image's last:
// the six windows are requested together. A pair that needs only 2 rows passes a third of weight 0.
template<int C, bool ODD>
__device__ __forceinline__ void AreaFixedTwoPairs(const uint8_t *rowA, const uint8_t *rowB, int srcRow, uint32_t at, uint32_t shift,
                                                  uint32_t rowBytes, uint32_t w01, uint32_t w23, const float (&wyA)[2][4],
                                                  const float (&wyB)[2][4], const float (&startA)[2], const float (&startB)[2],
                                                  uint32_t (&out)[4])
{
    uint32_t ra[3][C], rb[3][C];
#pragma unroll
    for (int j = 0; j < 3; ++j)
    {
        LoadQuadWindow<C, false, ODD>(rowA + (int64_t)j * srcRow, at, shift, false, rowBytes, ra[j]);
    }
#pragma unroll
    for (int j = 0; j < 3; ++j)
    {
        LoadQuadWindow<C, false, ODD>(rowB + (int64_t)j * srcRow, at, shift, false, rowBytes, rb[j]);
    }
    AreaSumRows<C, 3, 2>(ra, w01, w23, wyA, startA, &out[0]);
    AreaSumRows<C, 3, 2>(rb, w01, w23, wyB, startB, &out[2]);
}

template<int C, int K, bool GUARDED, bool ODD>
__device__ __forceinline__ void AreaFixedRowsOf(int n, const uint8_t *row, int srcRow, int lastRowIn, uint32_t at, uint32_t shift,
                                                uint32_t rowBytes, uint32_t w01, uint32_t w23, const float (&wy)[K][4],
                                                const float (&start)[K], uint32_t (&out)[K])
{
    // (wave-uniform)
    if (n == 3)
    {
        AreaFixedPixels<C, 3, K, GUARDED, ODD>(row, srcRow, lastRowIn, at, shift, rowBytes, w01, w23, wy, start, out);
    }
    else if (n == 2)
    {
        AreaFixedPixels<C, 2, K, GUARDED, ODD>(row, srcRow, lastRowIn, at, shift, rowBytes, w01, w23, wy, start, out);
    }
    else if (n == 4)
    {
        AreaFixedPixels<C, 4, K, GUARDED, ODD>(row, srcRow, lastRowIn, at, shift, rowBytes, w01, w23, wy, start, out);
    }
    else
    {
        AreaFixedPixels<C, 1, K, GUARDED, ODD>(row, srcRow, lastRowIn, at, shift, rowBytes, w01, w23, wy, start, out);
    }
}

// n source rows from `row` on; lastRowIn: which of them is the image's last row (n or more: none).
template<int C, int K, bool ODD>
__device__ __forceinline__ void AreaFixedRows(int n, const uint8_t *row, int srcRow, int lastRowIn, uint32_t at, uint32_t shift,
                                              uint32_t rowBytes, uint32_t w01, uint32_t w23, const float (&wy)[K][4],
                                              const float (&start)[K], uint32_t (&out)[K])
{
    if (C != 4 && lastRowIn < n) // wave-uniform, once per image and column tile
    {
        AreaFixedRowsOf<C, K, true, ODD>(n, row, srcRow, lastRowIn, at, shift, rowBytes, w01, w23, wy, start, out);
    }
    else
    {
        AreaFixedRowsOf<C, K, false, ODD>(n, row, srcRow, lastRowIn, at, shift, rowBytes, w01, w23, wy, start, out);
    }
}

// The tile of 64 columns x `rows` rows whose top left pixel is (x0, y0), both wave-uniform (y0 and rows multiples of 4).
template<int C, bool ODD>
__device__ __forceinline__ void ResizeAreaFixedWaveTile(const Plane &p, int x0, int y0, int rows)
{
    if (x0 >= p.dstW || y0 >= p.dstH)
    {
        return;
    }
    const int lane = threadIdx.x & 63;
    // columns and rows past the output compute a duplicate of the last one: every lane takes part in the transposes
    const int   dx = min(x0 + lane, p.dstW - 1);
    const float colStart = fminf(floorf(dx * p.scaleX), (float)(p.srcW - 4)); // the window never leaves its row
    float       cw[4];
    AreaWeights(p.scaleX, dx, p.srcW, 32768.f, colStart, false, cw);
    // rounding to an integer by adding 1.5 * 2^23: the low 16 bits of the sum's pattern are the integer
    uint32_t wq[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        wq[k] = __float_as_uint(cw[k] + 12582912.f);
    }
    const uint32_t w01 = __builtin_amdgcn_perm(wq[1], wq[0], 0x05040100u), w23 = __builtin_amdgcn_perm(wq[3], wq[2], 0x05040100u);
    const uint32_t off = (uint32_t)(int)colStart * C, at = C == 4 ? off : off & ~3u, shift = off & 3u;
    const uint32_t rowBytes = (uint32_t)p.srcW * C;

    // Row terms, lane l: output row y0 + (l & 15). Two vertically adjacent output rows (2i, 2i + 1) share the source
    // row between their boxes wherever the scale is not a whole number, so they are produced together from the
    // source rows first(2i) .. first(2i) + n - 1 when those are at most 4 (`pairRows`, else 0): `pw` are this row's
    // weights counted from first(2i). Otherwise each row on its own from its box's first row: `ow`, `ownRows`.
    const int   dy = min(y0 + (lane & (kAreaRowsMost - 1)), p.dstH - 1);
    const float ownStart = floorf(dy * p.scaleY), pairStart = floorf((dy & ~1) * p.scaleY);
    float       ow[4], pw[4];
    AreaWeights(p.scaleY, dy, p.srcH, 1.f / 32768.f, ownStart, true, ow);
    AreaWeights(p.scaleY, dy, p.srcH, 1.f / 32768.f, pairStart, true, pw);
    const int  ownRows = 1 + (ow[1] != 0.f) + (ow[2] != 0.f) + (ow[3] != 0.f);
    const bool fits    = fminf(dy * p.scaleY + p.scaleY, (float)p.srcH) <= pairStart + 4.f;
    const int  pairRows = !fits ? 0 : pw[3] != 0.f ? 4 : pw[2] != 0.f ? 3 : pw[1] != 0.f ? 2 : 1;
    const int  ownFirst = (int)ownStart, pairFirst = (int)pairStart;
    // the accumulator's start: minus 2^23 times the sum of the row's weights (see AreaRowSums), added in ascending order;
    // weights of 0 in front or behind change nothing, so the pair form and the single form start alike
    const float rowStart = -8388608.f * (((ow[0] + ow[1]) + ow[2]) + ow[3]);

    const int rowsHere = min(rows, p.dstH - y0);
    // output rows i, i + 1 -> out[0], out[1]
    auto rowPair = [&](int i, uint32_t *out)
    {
        const int n = __builtin_amdgcn_readlane(pairRows, i + 1);
        if (n != 0)
        {
            const int first = __builtin_amdgcn_readlane(pairFirst, i);
            float     wy[2][4];
            uint32_t  two[2];
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                wy[0][j] = ReadLane(pw[j], i);
                wy[1][j] = ReadLane(pw[j], i + 1);
            }
            const float start[2] = {ReadLane(rowStart, i), ReadLane(rowStart, i + 1)};
            AreaFixedRows<C, 2, ODD>(n, p.src + (int64_t)first * p.srcRow, p.srcRow, p.srcH - 1 - first, at, shift, rowBytes, w01,
                                w23, wy, start, two);
            out[0] = two[0];
            out[1] = two[1];
        }
        else
        {
#pragma unroll
            for (int k = 0; k < 2; ++k)
            {
                const int first = __builtin_amdgcn_readlane(ownFirst, i + k);
                float     wy[1][4];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    wy[0][j] = ReadLane(ow[j], i + k);
                }
                uint32_t    one[1];
                const float start[1] = {ReadLane(rowStart, i + k)};
                AreaFixedRows<C, 1, ODD>(__builtin_amdgcn_readlane(ownRows, i + k), p.src + (int64_t)first * p.srcRow, p.srcRow,
                                    p.srcH - 1 - first, at, shift, rowBytes, w01, w23, wy, start, one);
                out[k] = one[0];
            }
        }
    };
    // 4 output rows per step (rows past the output are duplicates of its last one and are not stored)
#pragma unroll 1
    for (int i = 0; i < rowsHere; i += 4)
    {
        uint32_t  q[1][4];
        const int nA = __builtin_amdgcn_readlane(pairRows, i + 1), nB = __builtin_amdgcn_readlane(pairRows, i + 3);
        const int firstA = __builtin_amdgcn_readlane(pairFirst, i), firstB = __builtin_amdgcn_readlane(pairFirst, i + 2);
        // the usual case at scales up to 1.5: both pairs from at most 3 rows each, clear of the image's last row
        // (wave-uniform)
        if (nA != 0 && nB != 0 && max(nA, nB) <= 3 && max(firstA, firstB) + 2 < p.srcH - 1)
        {
            float wyA[2][4], wyB[2][4];
#pragma unroll
            for (int j = 0; j < 3; ++j)
            {
                wyA[0][j] = ReadLane(pw[j], i);
                wyA[1][j] = ReadLane(pw[j], i + 1);
                wyB[0][j] = ReadLane(pw[j], i + 2);
                wyB[1][j] = ReadLane(pw[j], i + 3);
            }
            const float startA[2] = {ReadLane(rowStart, i), ReadLane(rowStart, i + 1)};
            const float startB[2] = {ReadLane(rowStart, i + 2), ReadLane(rowStart, i + 3)};
            AreaFixedTwoPairs<C, ODD>(p.src + (int64_t)firstA * p.srcRow, p.src + (int64_t)firstB * p.srcRow, p.srcRow, at, shift,
                                 rowBytes, w01, w23, wyA, wyB, startA, startB, q[0]);
        }
        else
        {
            rowPair(i, &q[0][0]);
            rowPair(i + 2, &q[0][2]);
        }
        StoreWavePatch<uint8_t, C>(p, x0, y0 + i, lane, q);
    }
}

// The same tile outside the fixed-point form's scales (image batches decide per image): one pixel at a time.
template<int C, bool VARSHAPE>
__device__ __forceinline__ void ResizeAreaPlainWaveTile(const Plane &p, int x0, int y0, int rows)
{
    const int dx = x0 + (int)(threadIdx.x & 63);
    if (dx >= p.dstW)
    {
        return;
    }
#pragma unroll 1
    for (int dy = y0; dy < min(y0 + rows, p.dstH); ++dy)
    {
        ResizePixel<uint8_t, C, NVCV_INTERP_AREA, VARSHAPE>(p, dx, dy);
    }
}

template<int C, bool ODD>
__global__ __launch_bounds__(256) void ResizeAreaFixedTensorKernel(const ResizeArgs a, const int rows, const WaveOrder order)
{
    const Plane p = GetPlanes<false>(a, blockIdx.z);
    const WaveTile t = WaveTileOf(order);
    ResizeAreaFixedWaveTile<C, ODD>(p, t.x * kAreaTileW, t.y * rows, rows);
}

template<int C, bool ODD>
__global__ __launch_bounds__(256) void ResizeAreaVarShapeKernel(const ResizeArgs a, const VarTiles tiles, const int rows)
{
    const TileCoord tc = LocateTile(tiles, blockIdx.x);
    const Plane     p  = GetPlanes<true>(a, tc.image);
    const int       x0 = tc.tx * kAreaTileW, y0 = (tc.ty * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * rows;
    if (AreaFixedDomain(p.scaleX, p.scaleY, p.srcW * C, p.srcH))
    {
        ResizeAreaFixedWaveTile<C, ODD>(p, x0, y0, rows);
    }
    else
    {
        ResizeAreaPlainWaveTile<C, true>(p, x0, y0, rows);
    }
}

// Bicubic for strong horizontal reductions. With one lane per output pixel the four taps of
// neighbouring lanes lie scale*pixel bytes apart, so each of a wave's tap loads touches 64 separate
// cache lines. Here the same 256 taps of a wave's row are fetched tap-major instead: lane l loads
// tap l%4 of pixel 16k + l/4 (k = 0..3), four lanes covering 4 contiguous pixels, and the wave
// hands the taps to their owners through LDS. Arithmetic and its order are those of ResizePixel.
// Bound by reading the source. `across`: the tiles of a row, where waves are counted along the rows, so that a block reads
// one long piece of each of its four source rows instead of short pieces of sixteen; 0: a block's waves are stacked, and
// find the source rows that they share in the L1. From a vertical scale of 4 on, where none are shared, the former is the
// faster one (16 x 4K f32x4 -> 640 x 360 268.9 -> 260.7 us, 5.7 TB/s; 21 x 344 x 1436 x 3 -> 76 x 304 23.9 -> 20.6; at 2.1, 1 x 3525 x
// 3205 x 4 -> 1665 x 1514, 40.4 -> 54.9; at 3.5, 1 x 6589 x 2303 x 4 -> 1553 x 668, 45.4 -> 47.2).
template<int BYTES>
struct alignas(BYTES % 16 == 0 ? 16 : (BYTES % 8 == 0 ? 8 : 4)) LdsSlot
{
    uint32_t w[BYTES / 4];
};

__device__ __forceinline__ void CubicSourceX(int srcW, float scaleX, int dx, int &sx, float &fx)
{
    const float cx = (dx + .5f) * scaleX - .5f;
    sx             = (int)floorf(cx);
    fx             = cx - sx;
    fx             = (sx < 1 || sx >= srcW - 3) ? 0.f : fx;
    sx             = max(1, min(sx, srcW - 3));
}

template<class T, int C>
__global__ __launch_bounds__(256) void ResizeCubicStagedKernel(const ResizeArgs a, const int across)
{
    using Px   = Pixel<T, C>;
    using Slot = LdsSlot<sizeof(Px)>;
    static_assert(sizeof(Px) % 4 == 0, "pixels are staged as whole dwords");
    __shared__ Slot stage[kTileH][kTileW * 4];

    const int   lane = threadIdx.x & 63;
    const int   wave = threadIdx.x >> 6; // (as a vector: 0.99 of the time, 301 launches)
    const Plane p    = GetPlanes<false>(a, blockIdx.z);
    int         tx = blockIdx.x, dy = blockIdx.y * kTileH + wave;
    if (across != 0)
    {
        const uint32_t along = blockIdx.x * 4u + (uint32_t)wave;
        dy                   = (int)(along / (uint32_t)across);
        tx                   = (int)along - dy * across;
    }
    const int dx = tx * kTileW + lane;

    const float scaleX = p.scaleX, scaleY = p.scaleY;

    // lanes and rows past the output compute a duplicate of the last pixel and skip the store: every
    // lane takes part in its wave's exchange (each wave owns one quarter of the staging array)
    int   sx;
    float fx;
    CubicSourceX(p.srcW, scaleX, min(dx, p.dstW - 1), sx, fx);
    const float cy = (min(dy, p.dstH - 1) + .5f) * scaleY - .5f;
    int         sy = (int)floorf(cy);
    const float fy = cy - sy;
    sy             = max(1, min(sy, p.srcH - 3));
    float wx[4], wy[4];
    CubicCoeffs(fx, wx);
    CubicCoeffs(fy, wy);

    // loader role: column of the tap this lane fetches in each of the four instructions
    int tapX[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        int   qsx;
        float qfx;
        CubicSourceX(p.srcW, scaleX, min(tx * kTileW + 16 * k + (lane >> 2), p.dstW - 1), qsx, qfx);
        tapX[k] = max(0, min(qsx - 1 + (lane & 3), p.srcW - 1));
    }

    Px   v[4][4];
    auto loadRow = [&](int j)
    {
        const int      yy  = max(0, min(sy - 1 + j, p.srcH - 1));
        const uint8_t *row = p.src + (int64_t)yy * p.srcRow;
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            v[j][k] = LoadPx<T, C>(row, tapX[k]);
        }
    };

    float sum[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        sum[c] = 0.f;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        loadRow(j);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            __builtin_memcpy(&stage[wave][64 * k + lane], &v[j][k], sizeof(Px));
        }
        WaveExchangeFence();
        Px t[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            __builtin_memcpy(&t[i], &stage[wave][4 * lane + i], sizeof(Px));
        }
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                sum[c] += (float)t[i].v[c] * (wx[i] * wy[j]);
            }
        }
        WaveExchangeFence();
    }
    if (dx < p.dstW && dy < p.dstH)
    {
        Px out;
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            out.v[c] = SaturateCast<T>(fabsf(sum[c]));
        }
        StorePx<T, C>(p.dst + (int64_t)dy * p.dstRow, dx, out);
    }
}

// ---------------------------------------------------------------------------------------------
// AREA of 8-bit pixels at reductions of more than the fixed-point form's 3 along an axis (up to kAreaWindowMost
// horizontally), tensors. Bound by reading the source. The sums are ResizeValue's, term by term in its order; what
// changes is how the source arrives. There a lane walks its box a few pixels per load and waits for each load in turn, and
// the launch takes the time of that chain. Here a row of the box is one window of K pixels from its first (partial or
// whole) pixel on, in up to three loads of 16 bytes from dword boundaries, and the windows of kAreaBatch rows are
// requested before the first is used (with windows a pixel wider, 3 rows: 39.7 us in the first case below, 4: 40.3, 6: 38.6, but 92 / 98 / 101 us in
// the second). Bytes of the window that are not whole pixels of the box are masked to 0, which a sum of non-negative terms
// does not notice, so every lane adds K pixels; the left partial pixel is the window's first, the right one is a load of its
// own (its place in the window differs from lane to lane); PARTIAL: the scale has such pixels. u8x3 32 x 1080p -> 320 x 180
// 56.6 -> 38.1 us (5.4 TB/s), 16 x 4K -> 500 x 281 176.5 -> 83 us, 32 x 1080p -> 571 x 323 142 -> 77 us, one 2363 x 1415 ->
// 355 x 153 15.9 -> 8.2 us; u8x4 16 x 4K -> 350 x 201 216 -> 117 us; u8x1 32 x 1080p -> 311 x 177 46.4 -> 24.9 us.
// REST: the rows that are left after whole batches are a batch of their own size, instead of one that asks for its last row
// again. Boxes whose rows are no multiple of 3 gain (4 x 720p u8x3 -> 492 x 180 7.4 -> 6.3 us, 2 x 4K u8x1 -> 549 x 1080 8.1 -> 7.0), but
// three and four channels pay with registers, so there it is for whole vertical scales alone (64 x 396 x 300 u8x3 -> 66 x 50
// 8.4 us without, 9.2 with it), of four channels at horizontal scales of more than 3 (64 x 400 x 296 -> 200 x 37 10.4 and 11.3; 16 x
// 720p -> 160 x 180 11.9 and 11.2); and one channel does without it where the boxes are whole batches (16 x 720p -> 160 x 240
// 6.2 and 6.5).
// Those figures are with windows a pixel wider at scales between whole numbers; as the dispatch has them now, 64 x 1283 x 721
// u8x3 -> 321 x 181 61.8 -> 52.9 us, -> 279 x 157 52.6 -> 50.1, -> 138 x 78 49.1 -> 45.0; u8x4 (48 images) 54.4 -> 46.1 us.
constexpr float kAreaWindowMost = 12.f;
constexpr int kAreaBatch = 3;

template<int C, int K>
struct AreaWindow
{
    static constexpr int kBytes = K * C, kDwords = (kBytes + 3) / 4; // brought to the front
    static constexpr int kLoad  = C == 4 ? K : (kBytes + 3 + 3) / 4;  // the dwords that hold them at any offset
    uint32_t d[kLoad];
    uint32_t right;
};

template<int C, int K, bool PARTIAL>
__device__ __forceinline__ void LoadAreaWindow(const uint8_t *row, uint32_t at, uint32_t rightAt, AreaWindow<C, K> &w)
{
    struct __attribute__((packed, aligned(1))) Dwords
    {
        uint32_t d[AreaWindow<C, K>::kLoad];
    };
    const Dwords v = *reinterpret_cast<const Dwords *>(row + at);
    __builtin_memcpy(w.d, &v, sizeof(v));
    if constexpr (PARTIAL)
    {
        w.right = C == 1 ? row[rightAt] : LoadU32Unaligned(row + rightAt);
    }
}

// The same for the image's last row, behind which nothing may be read: dwords that end behind the row are moved back.
template<int C, int K, bool PARTIAL>
__device__ __forceinline__ void LoadAreaWindowGuarded(const uint8_t *row, uint32_t at, uint32_t rightAt, uint32_t rowBytes,
                                                      AreaWindow<C, K> &w)
{
    auto dword = [&](uint32_t from)
    {
        const uint32_t back = min(from, rowBytes - 4), by = from - back;
        return by < 4 ? LoadU32Unaligned(row + back) >> (8 * by) : 0u;
    };
#pragma unroll
    for (int i = 0; i < AreaWindow<C, K>::kLoad; ++i)
    {
        w.d[i] = dword(at + 4 * i);
    }
    if constexpr (PARTIAL)
    {
        w.right = C == 1 ? row[rightAt] : dword(rightAt);
    }
}

template<int C, int K, bool PARTIAL, bool REST, int LANES>
__global__ __launch_bounds__(256) void ResizeAreaWindowKernel(const ResizeArgs a)
{
    using Window = AreaWindow<C, K>;
    const Plane p    = GetPlanes<false>(a, blockIdx.z);
    const int   lane = threadIdx.x & 63, dx = min((int)blockIdx.x * kTileW + lane, p.dstW - 1);
    const int   dy   = blockIdx.y * kTileH + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (dy >= p.dstH || (lane >= LANES && (int)blockIdx.x * kTileW + lane >= p.dstW))
    {
        return;
    }
    // (Of a tile with fewer columns LANES lanes work, those past the last column on it again. In a launch that leaves most of the chip idle a wave of 1 to 8
    // active lanes issues 2 to 3 times slower than one of more: a kernel of such sums alone, 26 blocks, 14.7 us with 9 to 64 lanes and 48 with
    // 1 to 8, 512 blocks no difference. One 640 x 480 u8x3 -> 66 x 50 15.1 -> 6.7 us, 500 x 480 -> 130 x 50 9.1 -> 5.1; 6 x 584 x 650 u8x4 -> 68 x 67
    // 18.1 -> 7.7. Time with 16 / 64 over that with the columns alone, 1200 launches: tiles of 1 to 8 columns, up to 64 blocks 0.73 / 0.69, 1024 0.94 / 0.94, more
    // 0.98 / 0.98; of 9 to 16, up to 64 0.98 / 0.91, more 1.00 / 0.99; of 17 to 63 0.99 / 0.99 up to 1024 blocks, in large launches 1.00 / 1.03. As an argument that a wave
    // waits for LANES costs 2 to 5 %.)
    // ResizeValue's terms; the vertical ones are the same in all lanes
    const float fsx1 = dx * p.scaleX, fsx2 = fsx1 + p.scaleX, fsy1 = dy * p.scaleY, fsy2 = fsy1 + p.scaleY;
    const int   xmin = (int)ceilf(fsx1), xmax = (int)floorf(fsx2);
    const int   ymin = __builtin_amdgcn_readfirstlane((int)ceilf(fsy1)), ymax = __builtin_amdgcn_readfirstlane((int)floorf(fsy2));
    const bool  hasLeft = xmin > fsx1, hasRight = xmax < fsx2 && xmax < p.srcW;
    const float scale = 1.f / (fminf(p.scaleX, p.srcW - fsx1) * fminf(p.scaleY, p.srcH - fsy1));
    const float left = hasLeft ? xmin - fsx1 : 0.f, right = hasRight ? fsx2 - xmax : 0.f;

    const uint32_t rowBytes = (uint32_t)p.srcW * C, off = (uint32_t)(xmin - (hasLeft ? 1 : 0)) * C;
    const uint32_t rightAt = (uint32_t)min(xmax, p.srcW - 1) * C;
    // whole pixels: bytes first .. last of the window
    const int first = hasLeft ? C : 0, last = first + (min(xmax, p.srcW) - xmin) * C;
    uint32_t  mask[Window::kDwords];
#pragma unroll
    for (int i = 0; i < Window::kDwords; ++i)
    {
        const int lo = min(max(first - 4 * i, 0), 4), hi = min(max(last - 4 * i, 0), 4);
        mask[i] = (uint32_t)((1ull << (8 * hi)) - (1ull << (8 * lo)));
        mask[i] = hi > lo ? mask[i] : 0u;
    }

    // rows in the order of the sums: the whole ones, the partial one above, the partial one below
    const int whole = max(min(ymax, p.srcH) - ymin, 0);
    const int above = ymin > fsy1 ? 1 : 0, below = ymax < fsy2 && ymax < p.srcH ? 1 : 0; // (uniform)
    const int rows  = __builtin_amdgcn_readfirstlane(whole + above + below);
    float     sum[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        sum[c] = 0.f;
    }
    [[maybe_unused]] auto addPixel = [&](uint32_t q, float w)
    {
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            sum[c] += (float)((q >> (8 * c)) & 0xFF) * w;
        }
    };
    // rows j0 .. j0 + B - 1
    auto addRows = [&](auto batch, int j0)
    {
        constexpr int B = decltype(batch)::value;
        Window        w[B];
        uint32_t      shift[B]; // of the window's first byte in its first dword (the low two bits)
#pragma unroll
        for (int b = 0; b < B; ++b)
        {
            const int j = REST ? j0 + b : min(j0 + b, rows - 1); // (a repeated row is not added)
            const int y = j < whole ? ymin + j : (j == whole && above ? ymin - 1 : ymax);
            const uint8_t *row = p.src + (int64_t)y * p.srcRow;
            if (y == p.srcH - 1)
            {
                LoadAreaWindowGuarded<C, K, PARTIAL>(row, off & ~3u, rightAt, rowBytes, w[b]);
                shift[b] = off;
            }
            else if constexpr (C == 4)
            {
                LoadAreaWindow<C, K, PARTIAL>(row, off, rightAt, w[b]);
            }
            else
            {
                // from the dword of memory that holds the first byte on
                const uint32_t mis = (uint32_t)reinterpret_cast<uintptr_t>(row) & 3u;
                shift[b]           = off + mis;
                LoadAreaWindow<C, K, PARTIAL>(row - mis, shift[b] & ~3u, rightAt + mis, w[b]);
            }
        }
#pragma unroll
        for (int b = 0; b < B; ++b)
        {
            const int j = j0 + b;
            if (!REST && j >= rows)
            {
                break;
            }
            const bool top = j == whole && above, bottom = j >= whole && !top;
            const float wy = top ? ymin - fsy1 : fsy2 - ymax; // (used for the partial rows only)
            const float wi = j < whole ? scale : wy * scale;
            const float wl = j < whole ? left * scale : wy * left * scale, wr = j < whole ? right * scale : wy * right * scale;
            uint32_t    r[Window::kDwords + 1];
#pragma unroll
            for (int i = 0; i < Window::kDwords; ++i)
            {
                r[i] = C == 4 ? w[b].d[i] : __builtin_amdgcn_alignbyte(w[b].d[min(i + 1, Window::kLoad - 1)], w[b].d[i], shift[b]);
            }
            [[maybe_unused]] const uint32_t px0 = r[0];
#pragma unroll
            for (int i = 0; i < Window::kDwords; ++i)
            {
                r[i] &= mask[i];
            }
#pragma unroll
            for (int k = 0; k < K; ++k)
            {
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    const int byte = k * C + c;
                    sum[c] += (float)((r[byte / 4] >> (8 * (byte % 4))) & 0xFF) * wi;
                }
            }
            if constexpr (PARTIAL)
            {
                if (bottom)
                {
                    addPixel(w[b].right, wr);
                    addPixel(px0, wl);
                }
                else
                {
                    addPixel(px0, wl);
                    addPixel(w[b].right, wr);
                }
            }
        }
    };
    int j0 = 0;
#pragma unroll 1
    for (; REST ? j0 + kAreaBatch <= rows : j0 < rows; j0 += kAreaBatch)
    {
        addRows(std::integral_constant<int, kAreaBatch>{}, j0);
    }
    if constexpr (REST)
    {
        static_assert(kAreaBatch == 3);
        if (rows - j0 == 2) // (uniform)
        {
            addRows(std::integral_constant<int, 2>{}, j0);
        }
        else if (rows - j0 == 1)
        {
            addRows(std::integral_constant<int, 1>{}, j0);
        }
    }
    Pixel<uint8_t, C> out;
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        out.v[c] = SaturateCast<uint8_t>(sum[c]);
    }
    if ((int)blockIdx.x * kTileW + lane < p.dstW)
    {
        StorePx<uint8_t, C>(p.dst + (int64_t)dy * p.dstRow, dx, out);
    }
}

// The kernel whose window holds a row of boxes `s` wide.
using AreaKernelPtr = void (*)(const ResizeArgs);

template<int C, bool PARTIAL, bool REST, int LANES>
AreaKernelPtr AreaWindowKernel(float s)
{
    return s <= 4.f   ? ResizeAreaWindowKernel<C, 4, PARTIAL, REST, LANES>
         : s <= 5.f   ? ResizeAreaWindowKernel<C, 5, PARTIAL, REST, LANES>
         : s <= 6.f   ? ResizeAreaWindowKernel<C, 6, PARTIAL, REST, LANES>
         : s <= 8.f   ? ResizeAreaWindowKernel<C, 8, PARTIAL, REST, LANES>
         : s <= 10.f  ? ResizeAreaWindowKernel<C, 10, PARTIAL, REST, LANES>
                      : ResizeAreaWindowKernel<C, 12, PARTIAL, REST, LANES>;
}

// Whether rows of the sources start at other places than dwords of memory, where a kernel has a form for that
// (LoadQuadWindow): any row of a tensor, any image of a batch.
template<int C>
bool RowsAreOdd(const ResizeArgs &a)
{
    return C != 4 && ((reinterpret_cast<uintptr_t>(a.srcBase) | (uint64_t)a.srcSampleStride | (uint32_t)a.srcRowStride) & 3) != 0;
}

template<int C>
bool RowsAreOdd(const NVCVImageBufferStrided *src, int count)
{
    return C != 4 && std::any_of(src, src + count, [](const NVCVImageBufferStrided &i)
                                 { return ((reinterpret_cast<uintptr_t>(i.planes[0].basePtr) | (uint32_t)i.planes[0].rowStride) & 3) != 0; });
}

// Where one lane per output pixel that walks its box is still the faster form: it reads four pixels per load, so boxes up to 2
// wide are one load a row, and boxes 4 and 8 wide have no rest. Its waves also hold fewer registers, which counts in large
// launches. us by pixels / by windows: boxes up to 2 wide and few rows high, 16 x 720p -> 853 x 180 u8x3 22.3 / 24.5, u8x4 21.8 / 26.7
// (one 640 x 480 of these, 210 blocks, 4.8 / 4.5 and 4.3 / 3.8; 4 x 720p u8x3 -> 674 x 225 9.5 / 8.9; 2 x 4K u8x4 -> 2258 x 240, 9 rows,
// 22.5 / 21.6); 4 wide, 16 x 720p -> 320 x 180 u8x3 9.6 / 10.4, -> 320 x 90 9.0 / 10.4, -> 320 x 288 11.0 / 11.1 (90 blocks, one 640 x
// 480 -> 160 x 120, 3.4 / 3.4); 8 wide, one 1080p -> 240 x 540 u8x3 3.4 / 4.0, u8x4 3.1 / 3.5, 16 x 720p -> 160 x 360 u8x4 13.0 / 11.7.
// One channel has no such sizes.
template<int C>
bool AreaPixelsAreFasterU8(const ResizeArgs &a, int64_t blocks)
{
    const float sx = a.scaleX, sy = a.scaleY;
    // (pixels of odd rows are not read four at a time at dwords: 16 x 1080p u8x3 -> 480 x 272 25.8 us, by windows 23.3)
    if (C == 3 && !RowsAreOdd<C>(a))
    {
        return (sx < 2.f && sx * sy <= 6.5f && blocks >= 4096)
            || (sx == 4.f && blocks >= 512 && (sy <= 2.f || sy >= 3.5f) && (sy <= 5.f || blocks >= 1360))
            || ((sx == 8.f || sx == 12.f) && sy <= 2.f && blocks >= 256);
    }
    return C == 4 && ((sx <= 2.f && sx * sy <= 8.5f && blocks >= 1024) || (sx == 8.f && sy == 2.f && blocks >= 256 && blocks < 1024));
}

// ---------------------------------------------------------------------------------------------
// AREA of float tensors at reductions of more than 1 along both axes (up to kAreaWindowMost horizontally). Bound by reading
// the source. With a lane walking its own box the lanes of a load lie a box apart, so every load touches all lines of the
// wave's part of the row, the L1 has lost them when the next pixel is asked for, and the L2 delivers the source as often as
// a box has columns. Here a wave that produces 64 columns of a row reads the boxes' rows 16 bytes per lane, whatever
// pixel they belong to, and sums them column by column in registers (KCHUNKS x 16 bytes per lane); the column sums
// then change lanes through LDS, and each lane adds those of its box. Sums of fewer terms each, so closer to the exact
// box filter (257 x 131 -> 214 x 109: 5.1e-8 of the norm, was 5.3e-8; 605 x 242 -> 55 x 22: 7.1e-8, was 1.6e-7). A column outside a lane's box is not
// added (not as 0 times itself, which an infinity would notice). 1283 x 721, 16 images f32x3: -> 1069 x 601 98.1 -> 70.5 us,
// -> 321 x 181 78.0 -> 40.1 (4.8 TB/s), -> 117 x 66 104 -> 41.1; 48 f32x1 -> 773 x 434 153 -> 92.9, -> 321 x 181 96.9 -> 45.7;
// 12 f32x4 -> 493 x 277 59.3 -> 40.6, -> 183 x 103 65.6 -> 35.1. (Each lane's own box as in the 8-bit form above, several
// rows ahead, asked the L1 for more lines at once: 0.5 to 1.9 times the speed of one pixel at a time.)
template<int C, int KCHUNKS>
__global__ __launch_bounds__(256) void ResizeAreaFloatKernel(const ResizeArgs a)
{
    typedef float F32x4 __attribute__((ext_vector_type(4)));
    typedef F32x4 UnalignedF32x4 __attribute__((aligned(4)));
    constexpr int kBatch = KCHUNKS <= 2 ? 4 : (KCHUNKS <= 5 ? 2 : 1); // rows in flight
    __shared__ float columns[4][KCHUNKS * 256];

    const Plane p    = GetPlanes<false>(a, blockIdx.z);
    const int   lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int   dx0 = blockIdx.x * kTileW, dx = min(dx0 + lane, p.dstW - 1), dy = blockIdx.y * kTileH + wave;
    if (dy >= p.dstH)
    {
        return;
    }
    const float fsx1 = dx * p.scaleX, fsx2 = fsx1 + p.scaleX, fsy1 = dy * p.scaleY, fsy2 = fsy1 + p.scaleY;
    // weights over the power of two above the box's size, so that no sum passes the largest value (exact: the last product
    // takes them out again)
    auto        above = [](float s) { return __uint_as_float((__float_as_uint(s) & 0x7f800000u) + (1u << 23)); };
    const float unitX = 1.f / above(p.scaleX), unitY = 1.f / above(p.scaleY);
    // the box's rows (uniform)
    const int yFirst = __builtin_amdgcn_readfirstlane((int)floorf(fsy1));
    const int yLast  = __builtin_amdgcn_readfirstlane(min((int)ceilf(fsy2), p.srcH) - 1);
    // the floats of a row from `base` to `end`, all that the boxes touch; lanes whose 4 would pass the end take the last 4
    const int base = min((int)floorf(dx0 * p.scaleX) * C, p.srcW * C - 4);
    const int last = max(min((int)ceilf(min(dx0 + kTileW, p.dstW) * p.scaleX) + 1, p.srcW) * C - 4, base);
    int       at[KCHUNKS];
    F32x4     sum[KCHUNKS];
#pragma unroll
    for (int i = 0; i < KCHUNKS; ++i)
    {
        at[i]  = min(4 * (lane + 64 * i), last - base);
        sum[i] = F32x4{0.f, 0.f, 0.f, 0.f};
    }
    const uint8_t *src = p.src + (int64_t)base * (int)sizeof(float);
#pragma unroll 1
    for (int y0 = yFirst; y0 <= yLast; y0 += kBatch)
    {
        F32x4 t[kBatch][KCHUNKS];
#pragma unroll
        for (int b = 0; b < kBatch; ++b)
        {
            const uint8_t *row = src + (int64_t)min(y0 + b, yLast) * p.srcRow; // (a repeated row is not added)
#pragma unroll
            for (int i = 0; i < KCHUNKS; ++i)
            {
                t[b][i] = *reinterpret_cast<const UnalignedF32x4 *>(row + (uint32_t)at[i] * 4u);
            }
        }
#pragma unroll
        for (int b = 0; b < kBatch; ++b)
        {
            const int y = y0 + b;
            if (y > yLast)
            {
                break;
            }
            const float wy = (fminf((float)(y + 1), fsy2) - fmaxf((float)y, fsy1)) * unitY;
#pragma unroll
            for (int i = 0; i < KCHUNKS; ++i)
            {
                sum[i] += t[b][i] * wy;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < KCHUNKS; ++i)
    {
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            columns[wave][at[i] + j] = sum[i][j]; // (lanes that took the same floats write the same sums)
        }
    }
    WaveExchangeFence();

    const float scale  = 1.f / (fminf(p.scaleX, p.srcW - fsx1) * fminf(p.scaleY, p.srcH - fsy1)) * (above(p.scaleX) * above(p.scaleY));
    const int   xFirst = (int)floorf(fsx1), xLast = min((int)ceilf(fsx2), p.srcW) - 1;
    const int   most   = (int)ceilf(p.scaleX) + 1; // columns that a box can touch
    float       out[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        out[c] = 0.f;
    }
#pragma unroll 1
    for (int k = 0; k < most; ++k)
    {
        const int    x  = min(xFirst + k, xLast);
        const float  wx = (fminf((float)(x + 1), fsx2) - fmaxf((float)x, fsx1)) * unitX;
        const float *q  = &columns[wave][x * C - base];
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            const float v = out[c] + q[c] * wx;
            out[c]        = xFirst + k <= xLast ? v : out[c];
        }
    }
    if (dx0 + lane < p.dstW)
    {
        Pixel<float, C> px;
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            px.v[c] = out[c] * scale;
        }
        StorePx<float, C>(p.dst + (int64_t)dy * p.dstRow, dx, px);
    }
}

// 16-byte pieces per lane that hold the columns of 64 boxes, those that edges between two columns add and one for their
// rounding; and the kernel for so many, of those that scales of more than 1 and up to kAreaWindowMost need (1 to 4, 1 to 10
// and 2 to 13 for 1, 3 and 4 channels).
template<int C>
constexpr int AreaFloatPieces(float scaleX)
{
    const float columns = scaleX * kTileW;
    const int   whole   = (int)columns;
    return ((whole + (columns > (float)whole ? 1 : 0) + 3) * C + 255) / 256;
}

// Boxes of few whole columns, where one lane per output pixel is still the faster form (it has no partial columns to add, and
// neighbouring lanes' boxes fill the lines they touch). One channel, whose pixels that form reads four at a time: 24 x 720p
// -> 320 x 180 15.0 us against 17.5 by column sums, one 4K -> 960 x 1440 8.4 and 10.5, -> 480 x 270 7.6 and 8.1 (one 720p ->
// 160 x 90, few blocks: 4.3 and 4.1), -> 1920 x 1080 10.4 and 11.1 (4 x 720p -> 640 x 360 5.8 and 5.7). Three and four channels
// while the memory-side cache holds the source: f32x4 one 720p -> 640 x 360 3.7 and 4.65, -> 320 x 180 4.5 and 5.2, 4 x 720p -> 640 x 553 16.1 and 17.2, but -> 320 x 480 20.5 and 16.4;
// 24 x 720p -> 640 x 553 95.7 and 86.1; f32x3 8 x 720p -> 640 x 553 23.4 and 26.6, one 720p -> 426 x 240 4.2 and 4.3.
template<int C>
bool AreaPixelsAreFaster(const ResizeArgs &a, int64_t blocks, int64_t srcBytes)
{
    const float s = a.scaleX;
    if constexpr (C == 1)
    {
        return s == 4.f || ((s == 5.f || s == 8.f) && blocks >= 512) || (s == 2.f && a.scaleY == 2.f && blocks >= 4096);
    }
    // (twice as wide and more than four times as high: 480p f32x3 -> 320 x 87 3.8 and 3.5, 4 x 720p -> 640 x 130 10.0 and 10.5;
    // three channels and partial rows: one 720p -> 640 x 232 4.54 and 4.21, 4 x 500 x 332 -> 250 x 107 4.6 and 4.4, whole ones
    // -> 640 x 360 3.7 and 4.06, -> 250 x 166 3.9 and 4.3)
    const bool rows = C == 4 || a.scaleY <= 2.f || std::ceil(a.scaleY) == a.scaleY;
    return s == 2.f ? srcBytes <= 128 << 20 && ((a.scaleY <= 4.f && rows) || srcBytes >= 32 << 20) : (s == 3.f || s == 4.f) && srcBytes <= 16 << 20;
}

using AreaFloatKernelPtr = void (*)(const ResizeArgs);

template<int C, int KCHUNKS = AreaFloatPieces<C>(kAreaWindowMost)>
AreaFloatKernelPtr AreaFloatKernel(int pieces)
{
    if constexpr (KCHUNKS > ((kTileW + 1 + 3) * C + 255) / 256)
    {
        if (pieces < KCHUNKS)
        {
            return AreaFloatKernel<C, KCHUNKS - 1>(pieces);
        }
    }
    return ResizeAreaFloatKernel<C, KCHUNKS>;
}

// ---------------------------------------------------------------------------------------------
// Bicubic resize of float tensors at scales below 2 along both axes. One pixel at a time the 16 taps of every
// output pixel are loaded and weighted, four fifths of them again for its neighbour below. Here a lane owns a column of
// `rows` output rows, forms each source row's weighted sum of four pixels once, keeps the last four of them and
// combines those for every output row between; the next source row is requested before the present rows are combined. Sums
// of four terms, twice, instead of sixteen: closer to the exact formula (131 x 97 -> 197 x 145: 6.2e-8 of the norm, was
// 7.7e-8). 4 x 1283 x 721
// f32x3 -> 1931 x 1081 64.9 -> 36.5 us (4.6 TB/s), -> 1200 x 700 27.3 -> 17.5, -> 963 x 541 19.6 -> 15.9; 2 x f32x4 -> 1280 x
// 960 21.6 -> 14.4; 12 x f32x1 -> 1931 x 1081 67.3 -> 51.7 (its writes: rows that start at no sector).
template<int C>
__global__ __launch_bounds__(256) void ResizeCubicStripF32Kernel(const ResizeArgs a, const int rows, const WaveOrder order)
{
    struct Taps
    {
        Pixel<float, C> px[4];
    };
    const Plane p    = GetPlanes<false>(a, blockIdx.z);
    const WaveTile tile = WaveTileOf(order);
    const int   lane = threadIdx.x & 63, dx = tile.x * kTileW + lane, y0 = tile.y * rows;
    if (y0 >= p.dstH)
    {
        return;
    }
    AxisTerms<4>   col = FinishedAxis<NVCV_INTERP_CUBIC>(p.scaleX, min(dx, p.dstW - 1), p.srcW, true);
    const uint32_t at  = (uint32_t)(col.s - 1) * (uint32_t)sizeof(Pixel<float, C>); // taps col.s - 1 .. col.s + 2, inside the row

    // Weights along a row add up to as much as 1.375 in magnitude, so a row of the type's extreme values would overflow
    // also where its own weight is 0. Halves here, doubled again with the row's weights (both exact).
    auto rowTerms = [&](int dy)
    {
        AxisTerms<4> r = FinishedAxis<NVCV_INTERP_CUBIC>(p.scaleY, dy, p.srcH, false);
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            r.w[i] *= 2.f;
        }
        return r;
    };
#pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        col.w[i] *= 0.5f;
    }

    auto load = [&](int y) { return *reinterpret_cast<const Taps *>(p.src + (int64_t)min(y, p.srcH - 1) * p.srcRow + at); };
    float h[4][C]; // halves of the sums of source rows first .. first + 3
    auto  rowSum = [&](const Taps &t, float (&out)[C])
    {
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            float v = t.px[0].v[c] * col.w[0];
            v += t.px[1].v[c] * col.w[1];
            v += t.px[2].v[c] * col.w[2];
            v += t.px[3].v[c] * col.w[3];
            out[c] = v;
        }
    };

    AxisTerms<4> row   = rowTerms(y0);
    int          first = __builtin_amdgcn_readfirstlane(row.s) - 1;
    {
        Taps t[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            t[j] = load(first + j);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            rowSum(t[j], h[j]);
        }
    }
    Taps      next = load(first + 4);
    const int yEnd = min(y0 + rows, p.dstH);
#pragma unroll 1
    for (int dy = y0;;)
    {
        Pixel<float, C> out;
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            float v = h[0][c] * row.w[0];
            v += h[1][c] * row.w[1];
            v += h[2][c] * row.w[2];
            v += h[3][c] * row.w[3];
            out.v[c] = fabsf(v);
        }
        if (dx < p.dstW)
        {
            StorePx<float, C>(p.dst + (int64_t)dy * p.dstRow, dx, out);
        }
        if (++dy >= yEnd)
        {
            break;
        }
        row              = rowTerms(dy);
        const int target = __builtin_amdgcn_readfirstlane(row.s) - 1;
#pragma unroll 1
        for (; first < target; ++first) // (up to twice; rows never go back)
        {
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                h[0][c] = h[1][c];
                h[1][c] = h[2][c];
                h[2][c] = h[3][c];
            }
            rowSum(next, h[3]);
            next = load(first + 5);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Bilinear resize of one-channel float pixels where rows are not reduced (maps and masks brought to their frames'
// size). Bound by the output's writes. Rows of such outputs rarely start at a multiple of 64 bytes (a dense row of 1917
// floats), and then every store instruction of a wave ends in two partly written 64-byte sectors that its neighbours
// complete in stores of their own: 3.78 M write requests where the output has 3.10 M sectors (24 x 513 x 289 ->
// 1917 x 1079). Writing alone, 199 MB in pieces of 30 KB to a block, takes 43.3 us where a wave's 1024 bytes start anywhere, 36.5 at
// 64-byte boundaries and 34.7 at 128-byte ones. So a block produces kRowsPerGroup whole rows (`groups` times, where one group does not give every wave a
// piece of 256 columns), collects them in LDS at the place they have relative to a 128-byte boundary and writes them
// out 16 bytes per lane on 16-byte boundaries: a dense output's rows as one run, whose two ends alone are partial. A
// lane's columns are 64 apart (LDS writes without bank conflicts); the tap pairs of all source rows that 4 output
// rows can need are requested before the first is used: 3, 4 or 5 by the scale. Against wave patches: 68.8 -> 44.1 us, 4.8 TB/s
// (24 x 513 x 289 -> 1917 x 1079), 22.8 -> 15.4 us (16 x 320 x 180 -> 1280 x 720), 13.9 -> 12.1 us (3 x 1901 x 900 -> 1300 x
// 1920). At 128-byte boundaries instead of 64-byte ones 41.3 -> 40.5 us (27 x 497 x 113 -> 2373 x 540 36.3 -> 35.0). The first case by other forms, each 3 to 4 us longer for an event behind every launch: this one 48.2 us, with 8 rows
// per group 61.6 us (61 KB of LDS leave two blocks per CU), streaming stores from the lanes that formed the values
// 53.5 us, cached stores, which the L2 merges to 3.13 M requests, 79 us (they evict the source rows).
constexpr int kRowsPerGroup = 4;

// Source rows from the first on that kRowsPerGroup output rows span, 3 to 5; 0: more than 5 (rows reduced). A place is
// a rounded product and a rounded difference, each off by at most 2^-11 below 8192: two of them by less than the margin.
static inline int LinearRowsSources(const ResizeArgs &a)
{
    const float span = (kRowsPerGroup - 1) * a.scaleY + (a.srcH == a.dstH ? 0.f : 4e-3f);
    return a.srcH > 8192 ? 0 : span <= 1.f ? 3 : span <= 2.f ? 4 : span <= 3.f ? 5 : 0;
}

template<int S>
__global__ __launch_bounds__(256) void ResizeLinearRowsKernel(const ResizeArgs a, const int chunks, const int groups)
{
    extern __shared__ __attribute__((aligned(16))) float stage[];
    const Plane p    = GetPlanes<false>(a, blockIdx.y);
    const int   lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int R  = kRowsPerGroup;
    const int   yBlock = blockIdx.x * groups * R, rowsBlock = min(groups * R, p.dstH - yBlock);
    // Row i of the block is staged from float i * pitch + lead(i) on, where lead is the row's distance from the 128-byte
    // boundary in front of it; dense rows follow one another in LDS as they do in memory (and keep the block's lead).
    const bool  dense = p.dstRow == 4 * p.dstW;
    const int   pitch = LinearRowsPitch(p.dstW, dense);
    auto        lead  = [&](int i)
    {
        return (int)(reinterpret_cast<uintptr_t>(p.dst + (int64_t)(yBlock + (dense ? 0 : i)) * p.dstRow) & 127) / 4;
    };
    for (int t = wave; t < chunks * groups; t += 4)
    {
        const int g = t / chunks, x0 = (t - g * chunks) * 256, y0 = yBlock + g * R;
        const int rows = min(R, p.dstH - y0);
        if (rows <= 0)
        {
            break;
        }
        float    wx1[4], wx0[4];
        uint32_t off[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            const float fx = (min(x0 + lane + 64 * k, p.dstW - 1) + .5f) * p.scaleX - .5f;
            const int   sx = (int)floorf(fx);
            wx1[k]         = sx < 0 ? 0.f : (sx > p.srcW - 2 ? 1.f : fx - sx);
            wx0[k]         = 1.f - wx1[k];
            off[k]         = (uint32_t)max(0, min(sx, p.srcW - 2)) * 4u;
        }
        const float fy = (min(y0 + min(lane, R - 1), p.dstH - 1) + .5f) * p.scaleY - .5f;
        const int   sy = (int)floorf(fy);
        const float wyLane = sy < 0 ? 0.f : (sy > p.srcH - 2 ? 1.f : fy - sy);
        const int   syLane = max(0, min(sy, p.srcH - 2));
        using Pair = Pixel<float, 2>;
        Pair          src[S][4];
        const int     first = __builtin_amdgcn_readlane(syLane, 0), last = __builtin_amdgcn_readlane(syLane, rows - 1) + 1;
#pragma unroll
        for (int i = 0; i < S; ++i)
        {
            const uint8_t *row = p.src + (int64_t)min(first + i, last) * p.srcRow;
#pragma unroll
            for (int k = 0; k < 4; ++k)
            {
                src[i][k] = *reinterpret_cast<const Pair *>(row + off[k]);
            }
        }
        int r = 0;
#pragma unroll
        for (int i = 0; i < S - 1; ++i)
        {
#pragma unroll 1
            for (; r < rows && __builtin_amdgcn_readlane(syLane, r) == first + i; ++r)
            {
                const float wy1 = ReadLane(wyLane, r), wy0 = 1.f - wy1;
                float      *to  = stage + (g * R + r) * pitch + lead(g * R + r) + x0 + lane;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                {
                    const float w00 = wx0[k] * wy0, w01 = wx1[k] * wy0, w10 = wx0[k] * wy1, w11 = wx1[k] * wy1;
                    const float v = src[i][k].v[0] * w00 + src[i][k].v[1] * w01 + src[i + 1][k].v[0] * w10 + src[i + 1][k].v[1] * w11;
                    if (x0 + lane + 64 * k < p.dstW)
                    {
                        to[64 * k] = v;
                    }
                }
            }
        }
    }
    __syncthreads();
    for (int run = 0; run < (dense ? 1 : rowsBlock); ++run)
    {
        const int    first = lead(run), end = first + (dense ? rowsBlock * p.dstW : p.dstW);
        const float *from = stage + run * pitch;
        uint8_t     *to   = p.dst + (int64_t)(yBlock + run) * p.dstRow - 4 * first;
        for (int i = threadIdx.x * 4; i < end; i += 1024)
        {
            uint32_t w[4];
            __builtin_memcpy(w, __builtin_assume_aligned(from + i, 16), 16);
            if (i >= first && i + 4 <= end)
            {
                StoreDwordsNT<4>(to + 4 * i, w);
            }
            else
            {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                {
                    if (i + k >= first && i + k < end)
                    {
                        *reinterpret_cast<uint32_t *>(to + 4 * (i + k)) = w[k];
                    }
                }
            }
        }
    }
}

// Which (type, channels, interpolation) run as wave patches.
template<class T, int C, int INTERP>
constexpr bool kPatchForm = INTERP != NVCV_INTERP_AREA && sizeof(Pixel<T, C>) <= 8;

template<class T, int C, int INTERP>
void LaunchTensor(const ResizeArgs &a, int N, hipStream_t stream)
{
    dim3 grid(DivUp(a.dstW, kTileW), DivUp(a.dstH, kTileH), N);
    if constexpr (INTERP == NVCV_INTERP_CUBIC && sizeof(Pixel<T, C>) % 4 == 0 && !kPatchForm<T, C, INTERP>)
    {
        if (a.srcW >= 2 * a.dstW)
        {
            const int  across = a.srcH >= 4 * (int64_t)a.dstH ? TilesAlongRows(a.dstW, a.dstH, kTileW) : 0;
            const dim3 sgrid  = across == 0 ? grid : dim3((unsigned)(((int64_t)across * a.dstH + 3) / 4), 1, N);
            hipLaunchKernelGGL((ResizeCubicStagedKernel<T, C>), sgrid, dim3(256), 0, stream, a, across);
            CheckLaunch("ResizeCubicStagedKernel");
            return;
        }
    }
    if constexpr (INTERP == NVCV_INTERP_CUBIC && std::is_same_v<T, float> && (C == 1 || C == 3 || C == 4))
    {
        // From a scale of 2 on a row sum serves one output row or two; a few waves leave their CUs idle in both forms, where a wave of one
        // row ends soonest (us as pixels / so, three channels: 224 x 224 -> 256 x 256 3.0 / 3.5, 320 x 240 -> 400 x 300 4.0 / 3.8; one
        // channel, the same: 3.7 / 3.1, 4.1 / 3.2; four channels reducing, 8 x 1050 x 93 -> 579 x 51, 1040 waves, 4.7 / 5.6, 3 x 1815 x 81 ->
        // 1012 x 43, 528, 3.6 / 4.4, 1 x 1550 x 121 -> 1480 x 115, 696, 3.8 / 4.0).
        auto waves = [&](int rows) { return (int64_t)DivUp(a.dstW, kTileW) * DivUp(a.dstH, rows) * N; };
        const int64_t least = C == 1 ? 128 : C == 4 && a.srcH > a.dstH ? (2 * (int64_t)a.srcH > 3 * (int64_t)a.dstH ? 2048 : 1024) : 512;
        if (a.srcW < 2 * (int64_t)a.dstW && a.srcH < 2 * (int64_t)a.dstH && a.srcW >= 4 && a.srcH >= 4 && waves(4) >= least)
        {
            // Rows per wave: a wave begins with four row sums. us with 4 / 8 / 16, three channels: 640 x 480 -> 800 x 600 4.8 / 5.1 / 7.3;
            // 8 x 256 x 256 -> 224 x 224 5.2 / 6.0 / 9.2; 32 of these 11.2 / 11.4 / 12.6; 720p -> 1080p 9.4 / 8.8 / 8.9; 2 x 1080p, as many, 21.2 /
            // 22.2 / 20.3; 4K 30.6 / 27.9 / 26.0; reducing, 4 x 1283 x 721 -> 963 x 541 15.8 / 17.0 / 16.1, four channels 20.3 / 21.5 / 19.4, one
            // 8.3 / 8.4 / 11.3. Enlarged rows that start at no line of memory are the better the sooner their neighbours follow (20 x 515
            // x 313 -> 815 x 460, 8 / 16, one channel 15.0 / 18.0, three 29.3 / 33.4, four 34.3 / 40.5; 12 x 1283 x 721 -> 1931 x 1081 39.8 / 53.0,
            // 112 / 118, 141 / 141), but not those that are about as many as the source's (four channels, 48 x 1461 x 42 -> 1478 x 42 22.8 / 19.3).
            const bool enlarging = a.srcH <= a.dstH, few = waves(8) <= 18 * 256 && (C == 1 || enlarging);
            const bool soon      = 5 * (int64_t)a.srcH <= 4 * (int64_t)a.dstH && a.dstRowStride % 64 != 0;
            const int  rows      = waves(4) <= 30 * 256 ? 4 : few || soon ? 8 : 16;
            // (along the rows where the chip is full, below one another, where rows share sources in the L1, before: one channel, 44 x 237 x 1008 -> 182 x
            // 962 30.2 -> 21.6, 65 x 569 x 51 -> 1915 x 128 26.4 -> 20.3; three, 11 x 793 x 146 -> 2918 x 454 54.8 -> 46.5, but 1 x 392 x 1105 -> 556 x 1567, 3528
            // waves of 4 rows, 6.4 and 7.3; four 44 x 286 x 59 -> 1071 x 223 48.6 and 42.5, but 128 x 104 x 88 -> 106 x 90 9.7 and 11.5. Not
            // three channels that share 4/5 of what is written: 189 x 424 x 66 -> 276 x 139 30.7 and 35.9, 1 x 955 x 1954 -> 521 x 4096 10.3 and 13.5, 33 launches up
            // to 4/3 1.04 times slower along the rows in the mean, from 1/4 to 2/3 0.97 to 0.98; one channel there 1.00.)
            const bool along     = C != 4 && rows > 4 && !(C == 3 && SharedRowsPay(a, kTileW, rows, 5, 4, 4));
            const auto order     = along ? AlongRows(a.dstW, a.dstH, kTileW, rows) : WaveOrder{};
            hipLaunchKernelGGL((ResizeCubicStripF32Kernel<C>), WaveTileGrid(a.dstW, a.dstH, N, kTileW, rows, order), dim3(256), 0, stream, a,
                               rows, order);
            CheckLaunch("ResizeCubicStripF32Kernel");
            return;
        }
    }
    // us as patches / in strips of 4 rows: 4 x 640 x 480 -> 1280 x 720 1 channel 4.4 / 4.2, 3 channels 6.4 / 5.6, 4 channels 5.3 / 5.0; one
    // 720p -> 1080p, 1080 strips of 8, 4.2 / 3.7, 4.6 / 4.8, 4.5 / 4.0; 16 x 160 x 160 -> 256 x 256, 512 of them, 3.9 / 3.6, 4.3 / 4.7, 4.0 / 3.8;
    // 4 x 224 x 224 -> 448 x 448, 448, 3.5 / 3.6, 3.8 / 4.5, 3.7 / 3.7.
    if constexpr (std::is_same_v<T, uint8_t> && INTERP == NVCV_INTERP_NEAREST && (C == 1 || C == 3 || C == 4))
    {
        const int64_t strips = (int64_t)DivUp(a.dstW, kQuadsTileW) * DivUp(a.dstH, kStripRows) * N;
        // Enlarged by less than 1.5 the patches, whose waves are a quarter as wide, are the faster form until the chip is full (us as
        // patches / so: 18 x 2140 x 137 x 1 -> 1089 x 98 4.2 / 5.0, 30 x 1219 x 75 x 1 -> 1201 x 78 4.4 / 5.0, 105 x 465 x 40 x 3 -> 576 x 50 5.3 / 6.9) and where most of a wave's 256 columns do not
        // exist (159 x 146 x 685 x 3 -> 53 x 361 9.7 / 13.8, 65 x 50 x 951 x 3 -> 64 x 1214 6.3 / 9.5; half of them, 18 x 514 x 1146 x 3 -> 558 x 1426, 22.0 / 17.4). 9 x 2475 x
        // 1391 x 1 -> 2801 x 1564 25.6 / 15.7; 39 x 830 x 212 x 3 -> 1054 x 366 22.7 / 16.4.
        const bool wide = C != 4 && a.srcW >= 24 && strips >= 10 * 256 && 5 * (int64_t)a.dstW >= 2 * (int64_t)DivUp(a.dstW, kQuadsTileW) * kQuadsTileW;
        if ((NearestStripScale<C>(a.srcW, a.srcH, a.dstW, a.dstH) && strips >= (C == 3 ? 6 : 4) * 256)
            || (wide && a.srcW <= a.dstW && a.srcH <= a.dstH))
        {
            // 4 rows: fewer registers, more waves in flight (8 / 4 rows: 8 x 720p -> 1080p 9.0 / 8.5, 15.3 / 13.6, 17.5 / 15.9; 32 x 224 x 224 ->
            // 448 x 448 6.1 / 5.3, 8.5 / 7.0, 9.4 / 7.2). One channel's largest launches pay more for the column terms (24 x 720p -> 1080p
            // 16.0 / 17.0, 32 of these 19.8 / 21.8) unless rows end inside lines of memory (100 x 300 x 300 -> 1000 x 500 20.5 / 18.7) and a
            // source row is fewer than three output rows (3 x 1336 x 1189 -> 3870 x 3444 13.4 / 15.5, 23 x 41 x 1275 -> 122 x 3819 9.3 / 10.5).
            const bool many   = 5 * (int64_t)a.dstH >= 11 * (int64_t)a.srcH ? strips >= 24 * 256 : strips >= 60 * 256 && a.dstRowStride % 64 == 0;
            const int  rows   = C == 1 && many ? kStripRows : 4;
            const auto order  = AlongRows(a.dstW, a.dstH, kQuadsTileW, rows);
            auto       kernel = rows == 4 ? ResizeNearestQuadsU8Kernel<C, 4> : ResizeNearestQuadsU8Kernel<C, C == 1 ? kStripRows : 4>;
            hipLaunchKernelGGL(kernel, WaveTileGrid(a.dstW, a.dstH, N, kQuadsTileW, rows, order), dim3(256), 0, stream, a, order);
            CheckLaunch("ResizeNearestQuadsU8Kernel");
            return;
        }
        if constexpr (C != 4)
        {
            if (wide && (C == 3 ? a.srcW <= a.dstW : a.srcW <= 4 * (int64_t)a.dstW))
            {
                // (a lane's 4 columns lie within 4 pixels of one channel more than the first one up to a scale of 4 / 3, 12 up to 4; within 3 of
                // three channels up to 1. Three channels reduced across, each pixel a load of its own: 143 launches from 0.83 to 1.27 of the patches' time)
                const auto order = AlongRows(a.dstW, a.dstH, kQuadsTileW, kNearestRows);
                auto kernel = C == 1 && 3 * (int64_t)a.srcW <= 4 * (int64_t)a.dstW ? ResizeNearestRowsU8Kernel<C, C == 1 ? 2 : 4>
                                                                                   : ResizeNearestRowsU8Kernel<C, 4>;
                hipLaunchKernelGGL(kernel, WaveTileGrid(a.dstW, a.dstH, N, kQuadsTileW, kNearestRows, order), dim3(256), 0, stream, a, order);
                CheckLaunch("ResizeNearestRowsU8Kernel");
                return;
            }
        }
    }
    if constexpr (kPairsForm<T, C, INTERP>)
    {
        if (a.srcW >= 4 && 3 * (int64_t)a.srcW <= 2 * (int64_t)a.dstW)
        {
            // Few waves run one round of loads and stores behind each other, so the launch's time is a wave's: shorter strips until
            // the chip is full (us with 8 / 4 / 2 rows, three channels: 224 x 224 -> 336 x 336 7.7 / 4.8 / 4.4; 4 x 224 x 224 -> 448 x
            // 448 8.2 / 6.6 / 5.2; 720p -> 1080p 8.8 / 6.9 / 7.2; 16 x 320 x 240 -> 640 x 480 11.4 / 11.2 / 11.2), from there on the
            // source rows that strips share and their column terms count (32 x 224 x 224 -> 448 x 448 12.2 / 13.0 / 13.2; one channel,
            // 8 x 720p -> 1080p 12.6 / 13.5 / 15.5).
            const int64_t strips = (int64_t)DivUp(a.dstW, kQuadsTileW) * DivUp(a.dstH, kStripRows) * N;
            const int     rows   = strips <= 3 * 256 ? 2 : strips <= 12 * 256 ? 4 : kStripRows;
            const auto    order  = FlatBlocks(a.dstW, kQuadsTileW) ? AlongRows(a.dstW, a.dstH, kQuadsTileW, rows) : WaveOrder{};
            auto          kernel = rows == 2   ? ResizeLinearQuadsU8Kernel<C, 2>
                                   : rows == 4 ? ResizeLinearQuadsU8Kernel<C, 4>
                                               : ResizeLinearQuadsU8Kernel<C, kStripRows>;
            hipLaunchKernelGGL(kernel, WaveTileGrid(a.dstW, a.dstH, N, kQuadsTileW, rows, order), dim3(256), 0, stream, a, order);
            CheckLaunch("ResizeLinearQuadsU8Kernel");
            return;
        }
        if (PairsFormScale<C>(a.srcW, a.dstW))
        {
            // Shorter strips while waves are few, as above (us with 4 / 2 rows, three channels: 720p -> 640 x 360 4.0 / 3.3; 15 x
            // 1136 x 166 -> 680 x 99 6.3 / 5.3; 32 x 256 x 256 -> 224 x 224 6.5 / 6.2, 64 of these 9.0 / 9.4; one channel, 4 x 720p ->
            // 960 x 540 5.0 / 5.0, 16 of these 11.2 / 12.5).
            const int64_t strips = (int64_t)DivUp(a.dstW, kPairsTileW) * DivUp(a.dstH, kPairStripRows) * N;
            const int     rows   = strips <= 16 * 256 ? 2 : kPairStripRows;
            const auto    order  = FlatBlocks(a.dstW, kPairsTileW) ? AlongRows(a.dstW, a.dstH, kPairsTileW, rows) : WaveOrder{};
            auto          kernel = rows == 2 ? ResizeLinearPairsU8Kernel<C, 2> : ResizeLinearPairsU8Kernel<C, kPairStripRows>;
            hipLaunchKernelGGL(kernel, WaveTileGrid(a.dstW, a.dstH, N, kPairsTileW, rows, order), dim3(256), 0, stream, a, order);
            CheckLaunch("ResizeLinearPairsU8Kernel");
            return;
        }
    }
    if constexpr (kAreaFixed<T, C, INTERP>)
    {
        if (AreaFixedDomain(a.scaleX, a.scaleY, a.srcW * C, a.srcH))
        {
            auto kernel = RowsAreOdd<C>(a) ? ResizeAreaFixedTensorKernel<C, C != 4> : ResizeAreaFixedTensorKernel<C, false>;
            const int rows = AreaRowsPerWave((int64_t)DivUp(a.dstW, kAreaTileW) * DivUp(a.dstH, kAreaRowsMost) * N);
            const auto order = AlongRows(a.dstW, a.dstH, kAreaTileW, rows);
            hipLaunchKernelGGL(kernel, WaveTileGrid(a.dstW, a.dstH, N, kAreaTileW, rows, order), dim3(256), 0, stream, a, rows, order);
            CheckLaunch("ResizeAreaFixedTensorKernel");
            return;
        }
    }
    if constexpr (kAreaFixed<T, C, INTERP>)
    {
        // Wider boxes than kAreaWindowMost, enlargements and rows shorter than a window keep the one-pixel form.
        if (a.scaleX > 1.f && a.scaleX <= kAreaWindowMost && a.scaleY > 1.f && a.srcW * C >= 64
            && !AreaPixelsAreFasterU8<C>(a, (int64_t)grid.x * grid.y * N))
        {
            // A box touches at most ceil(s) pixels per row besides the partial last one, which is not in the window: whole
            // scales s whole ones; between whole numbers floor(s) whole ones behind a partial first, or floor(s) + 1 without
            // one where the box's end rounds up (behind a partial first one it would have to round by more than the spacing
            // of the floats there).
            const bool partial = std::ceil(a.scaleX) != a.scaleX;
            const bool wholeY  = std::ceil(a.scaleY) == a.scaleY, batches = wholeY && std::fmod(a.scaleY, (float)kAreaBatch) == 0.f;
            const bool rest    = C == 1 ? !batches : wholeY && !batches && (C == 3 || a.scaleX > 3.f);
            const auto kernelOf = [&](auto lanes)
            {
                constexpr int L = decltype(lanes)::value;
                return partial ? (rest ? AreaWindowKernel<C, true, true, L>(a.scaleX) : AreaWindowKernel<C, true, false, L>(a.scaleX))
                               : (rest ? AreaWindowKernel<C, false, true, L>(a.scaleX) : AreaWindowKernel<C, false, false, L>(a.scaleX));
            };
            auto kernel = (int64_t)grid.x * grid.y * N <= 4 * 256 ? kernelOf(std::integral_constant<int, 64>{}) : kernelOf(std::integral_constant<int, 16>{});
            hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, a);
            CheckLaunch("ResizeAreaWindowKernel");
            return;
        }
    }
    if constexpr (INTERP == NVCV_INTERP_AREA && std::is_same_v<T, float> && (C == 1 || C == 3 || C == 4))
    {
        if (a.scaleX > 1.f && a.scaleX <= kAreaWindowMost && a.scaleY > 1.f && a.srcW >= 16
            && !AreaPixelsAreFaster<C>(a, (int64_t)grid.x * grid.y * N, (int64_t)a.srcW * a.srcH * C * 4 * N))
        {
            hipLaunchKernelGGL(AreaFloatKernel<C>(AreaFloatPieces<C>(a.scaleX)), grid, dim3(256), 0, stream, a);
            CheckLaunch("ResizeAreaFloatKernel");
            return;
        }
    }
    if constexpr (INTERP == NVCV_INTERP_CUBIC && std::is_same_v<T, uint8_t> && (C == 1 || C == 3 || C == 4))
    {
        constexpr int tileW = kCubicWalkW<C>;
        auto          waves = [&](int rows) { return (int64_t)DivUp(a.dstW, tileW) * DivUp(a.dstH, rows) * N; };
        // Fewer waves than 4 to a CU are left to the patches, whose waves are shorter (us as patches / so: 8 x 224 x 224 x 1 -> 256 x
        // 256 4.0 / 4.0, 100 x 100 x 3 -> 128 x 128 3.5 / 3.6; 640 x 480 x 3 -> 800 x 600 4.9 / 4.4). The farther the output rows are
        // apart, the less of a row's sums serve two of them, and the later it pays, in us as patches / in strips of 4 rows: 4 x 1209 x
        // 432 x 3 -> 448 x 160, 1120 waves, 4.6 / 5.0, 16 of these 8.0 / 8.0; from 1747 x 624 4.7 / 5.8 and 11.4 / 11.2, in strips of 8 12.2;
        // 12 x 1728 x 972 x 3 -> 640 x 360, in strips of 8, 15.2 / 14.1. Four channels: 4 x 1747 x 624 -> 448 x 160 4.7 / 5.0, 6 x 2496 x
        // 1404 -> 640 x 360 16.3 / 15.6. One: 1024 to 1536 waves, at a scale of 2, 3 to 10 % more as strips, from 1536 on 8 % less. Where a quarter of the
        // lanes have no column it does not pay at these scales (51 x 481 x 723 x 1 -> 257 x 387 14.6 / 17.7; 33 x 405 x 1099 x 3 -> 133 x
        // 362, in strips of 8, 13.7 / 16.2).
        const bool    over2 = a.srcH > 2 * (int64_t)a.dstH, reducing = a.srcH > a.dstH;
        const bool    far   = C == 1 ? 4 * (int64_t)a.srcH > 7 * (int64_t)a.dstH : C == 3 ? over2 : a.srcH > 3 * (int64_t)a.dstH;
        const int64_t least = !far ? 4 : C == 1 ? 6 : C == 3 ? 32 : 16;
        const bool    idle  = C != 4 && far && 4 * (int64_t)a.dstW < 3 * (int64_t)DivUp(a.dstW, tileW) * tileW;
        if (CubicWalks<C>(a.srcW, a.srcH, a.dstW, a.dstH) && waves(4) >= least * 256 && !idle)
        {
            // A wave's first row costs three row sums more than the others, its end leaves the CU to fewer waves. us with 4 / 8 / 16 / 32
            // rows, enlarging: 1280 x 720 x 3 -> 1080p 7.6 / 6.8 / 7.4 / 10.8; 6 x 576 x 324 x 4 -> 640 x 360 5.7 / 6.1 / 7.2; 21 x 1119 x
            // 343 x 3 -> 1140 x 403 27.2 / 21.7 / 20.6 / 23.1; 32 x 1280 x 720 x 3 -> 1080p 139 / 101 / 87 / 79. Reducing, where a strip has
            // more row sums to each output row: 4 x 896 x 503 x 3 -> 640 x 360 5.7 / 6.5 / 8.6, 8 of these 7.5 / 8.1 / 10.0, 24 of these
            // 16.3 / 14.4 / 15.9; 64 x 256 x 256 x 3 -> 224 x 224 12.1 / 10.6 / 11.6 / 14.9; 64 x 627 x 224 x 3 -> 448 x 160 16.4 / 14.5 / 15.0; by
            // more than 2 the rows of four channels are what the launch reads, 6 x 1728 x 972 x 4 -> 640 x 360 10.7 / 10.0 / 13.0. One
            // channel, whose waves are four times as wide: 8 x 2560 x 720 -> 1280 x 360, 3600 waves of 4 rows, 8.3 / 7.7 / 9.7. 32 only where the
            // lines of memory that output rows end in are not shared with a neighbour that comes to them late (9 x 1515 x 649 x 3 -> 3815 x
            // 1860, 16 / 32: 74 / 90).
            int rows = 4;
            rows     = waves(8) >= (C == 1 ? 6 : C == 4 && over2 ? 8 : reducing ? 16 : 10) * 256 ? 8 : rows;
            rows     = waves(16) >= (C == 3 ? 20 : 16) * 256 ? 16 : rows;
            rows     = waves(32) >= 64 * 256 && a.dstH > a.srcH && a.dstRowStride % 64 == 0 ? 32 : rows;
            const auto    order = AlongRows(a.dstW, a.dstH, tileW, rows);
            constexpr int kTwo = C == 1 ? 2 : 1;
            auto kernel = C == 1 ? (10 * (int64_t)a.srcW <= 13 * (int64_t)a.dstW ? ResizeCubicWalkU8Kernel<C, 1, false> : ResizeCubicWalkU8Kernel<C, kTwo, false>)
                                 : (RowsAreOdd<C>(a) ? ResizeCubicWalkU8Kernel<C, 1, C == 3> : ResizeCubicWalkU8Kernel<C, 1, false>);
            hipLaunchKernelGGL(kernel, WaveTileGrid(a.dstW, a.dstH, N, tileW, rows, order), dim3(256), 0, stream, a, rows, order);
            CheckLaunch("ResizeCubicWalkU8Kernel");
            return;
        }
    }
    if constexpr (std::is_same_v<T, float> && C == 1 && INTERP == NVCV_INTERP_LINEAR)
    {
        const int sources = LinearRowsSources(a), chunks = DivUp(a.dstW, 256);
        const int groups = chunks >= 3 ? 1 : chunks == 2 ? 2 : 4;
        const int lds = LinearRowsLds(a.dstW, a.dstRowStride == 4 * (int64_t)a.dstW, groups * kRowsPerGroup);
        const dim3 rgrid(DivUp(a.dstH, groups * kRowsPerGroup), N);
        const int64_t blocks = (int64_t)rgrid.x * N;
        // us as patches / as rows:
        // - Close to three blocks and more per CU: below that the wave patches spread further (one 513 x 289 -> 1917 x 1079, 270
        //   blocks: 5.3 / 6.3; 3 x 1281 x 721, 543: 7.0 / 7.9; 4 x 1026 x 578, 580: 5.9 / 6.5; 4 x 1281 x 721, 724: 8.8 / 8.2).
        // - Rows that fill a wave's 256 columns well: 2929 x 64 x 64 18.0 / 29.7; 244 x 128 x 128 7.7 / 8.3, from 64 x 64 7.2 / 7.1,
        //   732 of these 17.5 / 14.9; 156 x 160 x 160 8.4 / 7.8.
        // - Three blocks per CU and more in the LDS (one 1080p -> 4K, two per CU: 13.2 / 19.7, 4 of these 45.6 / 49.3; 4 maps of 3100 rows of
        //   3352 floats, the last of three: 51.5 / 47.7, of 3355 floats: 54.0 / 62.3), and with
        //   three no second round of blocks that is nearly empty (2 x 2560 x 1440, 720 blocks for 768 places: 12.3 / 10.6; 2 x
        //   2816 x 1584, 792: 14.9 / 17.2; 4 of these 26.6 / 26.0). 3 maps of 2000 rows of 2513 floats, four per CU: 22.2 / 19.7.
        const bool wide   = a.dstW >= 144 || (a.dstW >= 96 && a.dstW >= 2 * a.srcW && (int64_t)a.dstW * a.dstH * N >= 4000000);
        const int  perCu  = BlocksPerCu(lds);
        const bool rounds = perCu >= 4 || (perCu == 3 && (blocks <= 3 * 256 || blocks >= 6 * 256));
        if (sources != 0 && a.srcW >= 2 && a.srcH >= 2 && blocks >= 704 && wide && rounds)
        {
            auto kernel = sources == 3 ? ResizeLinearRowsKernel<3> : sources == 4 ? ResizeLinearRowsKernel<4> : ResizeLinearRowsKernel<5>;
            hipLaunchKernelGGL(kernel, rgrid, dim3(256), lds, stream, a, chunks, groups);
            CheckLaunch("ResizeLinearRowsKernel");
            return;
        }
    }
    if constexpr (kPatchForm<T, C, INTERP>)
    {
        // a launch of under 8 four-wave blocks per CU is spread as single-wave blocks: it is latency-bound
        // and finishes sooner the more CUs take part
        const int64_t blocks = (int64_t)DivUp(a.dstW, kPatchTileW) * DivUp(a.dstH, kPatchTileH) * N;
        const int     waves  = blocks < 8 * 256 ? 1 : 4;
        // (Below one another where rows share much more than they write. Bicubic f32x1 from 4/3 on: 105 x 1100 x 213 -> 336 x 461 61.0 and along the rows 74.1, 9 x
        // 797 x 345 -> 296 x 923 9.8 and 12.5, 42 launches 1.05 to 1.29 times slower so, 1.02 to 1.17 with inputs out of the memory's cache; less shared 0.96 to 1.01.
        // u8x4 from 5/3 on: 4 x 1223 x 1985 -> 447 x 3990 15.5 and 17.2, 105 x 1100 x 213 -> 336 x 461 31.6 and 35.6, 22 launches 1.05, out of the cache 1.00; less 0.96
        // to 1.00. Smaller pixels and bilinear f32x1: 0.98 to 1.00.)
        constexpr bool kCubicF = std::is_same_v<T, float> && C == 1 && INTERP == NVCV_INTERP_CUBIC,
                       kLinear4 = std::is_same_v<T, uint8_t> && C == 4 && INTERP == NVCV_INTERP_LINEAR;
        const bool shared = waves == 4 && ((kCubicF && SharedRowsPay(a, kPatchTileW, 4, 3, 4, 8)) || (kLinear4 && SharedRowsPay(a, kPatchTileW, 4, 3, 5, 4)));
        const auto order = shared ? WaveOrder{} : AlongRows(a.dstW, a.dstH, kPatchTileW, 4);
        constexpr bool kOdd   = INTERP == NVCV_INTERP_CUBIC && kFixedCubic<T> && C != 4;
        auto           kernel = kOdd && RowsAreOdd<C>(a) ? ResizePatchTensorKernel<T, C, INTERP, kOdd> : ResizePatchTensorKernel<T, C, INTERP, false>;
        hipLaunchKernelGGL(kernel, WaveTileGrid(a.dstW, a.dstH, N, kPatchTileW, 4, order, waves),
                           dim3(64 * waves), 0, stream, a, order);
        CheckLaunch("ResizePatchTensorKernel");
        return;
    }
    // Enlarging, the launch's time is its writes and a block that writes one run of a row is faster (8 x 720p -> 1080p
    // f32x3 bilinear 56.4 -> 45.5 us, f32x4 68.1 -> 56.3 us); reducing, it is the reads, and the four rows of the
    // 64 x 4 block share source rows (1080p -> 720p f32x3 bilinear 41.1 us against 49.3 us flat).
    // (bicubic keeps the 64 x 4 block: its time is the arithmetic's and did not change with the block)
    // (Nearest neighbour shares no source rows but with itself: 76 x 107 x 227 f32x3 -> 66 x 140 6.9 -> 5.6 us, 65 x 80 x 82 -> 307 x 314 18.5 -> 15.4, 104 x
    // 46 x 743 f32x4 -> 65 x 1048 36.8 -> 31.1. Enlarged down by 4/3 and more it shares enough to keep the 64 x 4 block where output rows end with a sector of
    // memory and fill the waves to 80 % (block / along the rows: 107 x 140 x 35 x 4 -> 436 x 152 20.3 / 24.5, 38 x 146 x 90 x 4 -> 556 x 383 21.5 / 25.1; 172
    // launches of f32x4 and 47 of f32x3, 2 to 9 % and 2 to 6 % in the mean of their classes). Where they do not, along the rows is the faster one, by up to 10 %, unless what
    // is shared is half of what is written or more: 168 x 1115 x 34 x 3 -> 375 x 130 36.0 / 54.1, 6 x 1176 x 470 x 3 -> 475 x 1211 14.8 / 22.3, 10 x 530 x 137 x 4 -> 204 x
    // 496 5.7 / 9.0; 86 launches of f32x3 1.17 times slower along the rows in the mean, 1.08 with inputs that are not in the memory's cache, 79 of f32x4 1.12 and 1.07;
    // 96 whose waves are filled to 70 .. 80 % 1.11 and 1.07, to 60 .. 70 % 1.02 and 1.01, less 0.89 and 0.95; less shared, from 1/4 to 1/2, 0.98 to 1.00.)
    // (Bilinear rows share theirs with the next one below a vertical scale of 2: 20 x 722 x 418 f32x3 -> 836 x
    // 484 33.9 us in the 64 x 4 block and 40.7 along the rows, 12 x 399 x 367 f32x4 -> 534 x 492 14.9 and 19.2; at 2.8, 121 x 194 x 594 f32x3 -> 69 x 211,
    // 31.2 and 25.4.)
    // Enlarged rows of 1024 pixels and more start with a block, where they are not counted along the rows: 4 x 720p -> 1080p f32x3 nearest neighbour 22.7 so, 23.7
    // along the rows, 24.6 in the 64 x 4 block; but 16 bytes to a pixel keep that block, 39 launches at 0.90 to 0.95 of the time in the mean, and so do nearest
    // neighbour's 12 unless a row has a multiple of 8 blocks, which puts a column's rows on one XCD (there 0.79 of the time along the rows, 0.93 in the 64 x 4
    // block, 73 launches; others 0.73 to 1.27 and 0.68 to 0.82 in their means, 4 x 6565 x 24 -> 2113 x 153 5.5 along the rows, 10.7 so).
    const bool shared = (4 * (int64_t)a.srcH <= 3 * (int64_t)a.dstH && a.dstRowStride % 64 == 0
                         && 4 * (int64_t)DivUp(a.dstW, kTileW) * kTileW <= 5 * (int64_t)a.dstW)
                     || SharedRowsPay(a, kTileW, 1, 2, 1, 10, 70);
    const bool along = INTERP == NVCV_INTERP_NEAREST ? !shared : INTERP == NVCV_INTERP_LINEAR && a.srcH >= 2 * (int64_t)a.dstH;
    const bool flat  = INTERP != NVCV_INTERP_CUBIC && (INTERP != NVCV_INTERP_NEAREST || (sizeof(Pixel<T, C>) < 16 && DivUp(a.dstW, 4 * kTileW) % 8 == 0))
                    && (int64_t)a.dstW * a.dstH > (int64_t)a.srcW * a.srcH && FlatBlocks(a.dstW, kTileW);
    const auto order = along ? AlongRows(a.dstW, a.dstH, kTileW, 1)
                     : flat  ? AlongRows(DivUp(a.dstW, 4 * kTileW) * 4 * kTileW, a.dstH, kTileW, 1)
                             : WaveOrder{};
    hipLaunchKernelGGL((ResizeTensorKernel<T, C, INTERP>), WaveTileGrid(a.dstW, a.dstH, N, kTileW, 1, order), dim3(256), 0, stream, a, order);
    CheckLaunch("ResizeTensorKernel");
}

template<class T, int C, int INTERP>
void LaunchVarShape(const ResizeArgs &a, const NVCVImageBufferStrided *srcHost, const NVCVImageBufferStrided *dstHost, int N,
                    hipStream_t stream)
{
    for (int first = 0; first < N; first += kMaxTileImages)
    {
        VarTiles  tiles;
        const int count = std::min(kMaxTileImages, N - first);
        // whether most output pixels of this launch lie in images for which a block of four waves side by side pays
        // (FlatBlocks), given a wave's tile; and the block's tile either way
        auto flatFor = [&](int waveW)
        {
            int64_t flatPixels = 0, allPixels = 0;
            for (int i = first; i < first + count; ++i)
            {
                const int64_t px = (int64_t)dstHost[i].planes[0].width * dstHost[i].planes[0].height;
                allPixels += px;
                flatPixels += FlatBlocks(dstHost[i].planes[0].width, waveW) ? px : 0;
            }
            return 2 * flatPixels > allPixels;
        };
        auto buildTiles = [&](int waveW, int waveH, bool flat)
        { return BuildVarTiles(tiles, dstHost, first, count, flat ? 4 * waveW : waveW, flat ? waveH : 4 * waveH); };
        if constexpr (kPairsForm<T, C, INTERP>)
        {
            // strips when that still gives every CU 8 blocks: the wide tile where most output pixels belong to images
            // that take four columns per lane
            int64_t quadPixels = 0, allPixels = 0;
            for (int i = first; i < first + count; ++i)
            {
                const int64_t px = (int64_t)dstHost[i].planes[0].width * dstHost[i].planes[0].height;
                allPixels += px;
                quadPixels += QuadStripScale<C>(srcHost[i].planes[0].width, dstHost[i].planes[0].width) ? px : 0;
            }
            bool flat  = flatFor(kStripsWaveW<true>);
            int  total = 2 * quadPixels > allPixels ? buildTiles(kStripsWaveW<true>, kStripsWaveH<true>, flat) : 0;
            if (total >= 8 * 256)
            {
                hipLaunchKernelGGL((ResizeLinearStripsU8VarShapeKernel<C, true>), dim3(total), dim3(256), 0, stream, a, tiles, (int)flat);
                CheckLaunch("ResizeLinearStripsU8VarShapeKernel");
                continue;
            }
            flat  = flatFor(kStripsWaveW<false>);
            total = buildTiles(kStripsWaveW<false>, kStripsWaveH<false>, flat);
            if (total >= 8 * 256)
            {
                hipLaunchKernelGGL((ResizeLinearStripsU8VarShapeKernel<C, false>), dim3(total), dim3(256), 0, stream, a, tiles, (int)flat);
                CheckLaunch("ResizeLinearStripsU8VarShapeKernel");
                continue;
            }
            total = BuildVarTiles(tiles, dstHost, first, count, kPairsTileW, kPairsTileH);
            if (total > 0)
            {
                hipLaunchKernelGGL((ResizeLinearPairsU8VarShapeKernel<C>), dim3(total), dim3(256), 0, stream, a, tiles);
                CheckLaunch("ResizeLinearPairsU8VarShapeKernel");
            }
            continue;
        }
        if constexpr (kAreaFixed<T, C, INTERP>)
        {
            int       total = BuildVarTiles(tiles, dstHost, first, count, kAreaTileW, 4 * kAreaRowsMost);
            const int rows  = AreaRowsPerWave(4 * (int64_t)total);
            if (rows != kAreaRowsMost)
            {
                total = BuildVarTiles(tiles, dstHost, first, count, kAreaTileW, 4 * rows);
            }
            if (total > 0)
            {
                auto kernel = RowsAreOdd<C>(srcHost + first, count) ? ResizeAreaVarShapeKernel<C, C != 4> : ResizeAreaVarShapeKernel<C, false>;
                hipLaunchKernelGGL(kernel, dim3(total), dim3(256), 0, stream, a, tiles, rows);
                CheckLaunch("ResizeAreaVarShapeKernel");
            }
            continue;
        }
        if constexpr (INTERP == NVCV_INTERP_NEAREST && std::is_same_v<T, uint8_t> && (C == 1 || C == 3 || C == 4))
        {
            int64_t stripPixels = 0, allPixels = 0;
            for (int i = first; i < first + count; ++i)
            {
                const NVCVImagePlaneStrided &sp = srcHost[i].planes[0], &dp = dstHost[i].planes[0];
                const int64_t                px = (int64_t)dp.width * dp.height;
                allPixels += px;
                stripPixels += NearestStripScale<C>(sp.width, sp.height, dp.width, dp.height) ? px : 0;
            }
            const bool flat  = flatFor(kStripsWaveW<true>);
            // (us as patches / 4 rows, three channels: 8 x 640 x 480 -> 1280 x 720 10.8 / 8.0; 32 x 224 x 224 -> 448 x 448 9.8 / 7.1; 8 x
            // 320 x 240 -> 640 x 480 5.8 / 5.9; 8 / 4 rows: 16 x 720p -> 1080p 24.2 / 20.9, one channel 13.8 / 16.1)
            if (2 * stripPixels > allPixels)
            {
                int rows  = C == 1 ? kStripRows : 4;
                int total = buildTiles(kStripsWaveW<true>, rows, flat);
                if (C == 1 && total < 8 * 256)
                {
                    rows  = 4;
                    total = buildTiles(kStripsWaveW<true>, rows, flat);
                }
                if (total >= 2 * 256)
                {
                    auto kernel = rows == 4 ? ResizeNearestStripsU8VarShapeKernel<C, 4> : ResizeNearestStripsU8VarShapeKernel<C, C == 1 ? kStripRows : 4>;
                    hipLaunchKernelGGL(kernel, dim3(total), dim3(256), 0, stream, a, tiles, (int)flat);
                    CheckLaunch("ResizeNearestStripsU8VarShapeKernel");
                    continue;
                }
            }
        }
        if constexpr (INTERP == NVCV_INTERP_CUBIC && std::is_same_v<T, uint8_t> && (C == 3 || C == 4))
        {
            // walked where most output pixels belong to images that can be and every CU still gets 8 blocks (us as patches / so, images
            // of sizes up to 10 % about these, three channels: 128 x 256 x 256 -> 224 x 224, 2048 blocks, 28.0 / 26.7, 64 of these 15.9 /
            // 16.0; 16 x 640 x 480 -> 800 x 600, 2140, 27.9 / 24.1, 4 of these 9.9 / 11.1; 8 x 1080p -> 720p, 2041, 29.1 / 28.7, 4 of these
            // 17.6 / 19.8; 24 x 1000 x 700 -> 400 x 300, 835, 16.6 / 22.6; four channels 27.4 / 23.2 and 15.8 / 13.7, 30.1 / 23.1 and 10.2 /
            // 10.4, 31.1 / 27.7 and 18.3 / 17.5, 19.0 / 19.2). 16 rows a wave: with 8 / 16 / 32 16 x 640 x 480 -> 800 x 600 25.0 / 24.1 / 26.2, 32 x
            // 1080p -> 720p 102 / 94 / 93, 32 x 720p -> 1080p 157 / 137 / 128.
            int64_t walked = 0, all = 0;
            for (int i = first; i < first + count; ++i)
            {
                const NVCVImagePlaneStrided &in = srcHost[i].planes[0], &out = dstHost[i].planes[0];
                const int64_t                px = (int64_t)out.width * out.height;
                all += px;
                walked += CubicWalks<C>(in.width, in.height, out.width, out.height) ? px : 0;
            }
            int total = 2 * walked > all ? BuildVarTiles(tiles, dstHost, first, count, kPatchTileW, 4 * kCubicBatchRows) : 0;
            if (total >= 8 * 256)
            {
                auto kernel = RowsAreOdd<C>(srcHost + first, count) ? ResizeCubicWalkU8VarShapeKernel<C, C != 4>
                                                                    : ResizeCubicWalkU8VarShapeKernel<C, false>;
                hipLaunchKernelGGL(kernel, dim3(total), dim3(256), 0, stream, a, tiles);
                CheckLaunch("ResizeCubicWalkU8VarShapeKernel");
                continue;
            }
        }
        if constexpr (kPatchForm<T, C, INTERP>)
        {
            const bool flat  = flatFor(kPatchTileW);
            int        total = buildTiles(kPatchTileW, 4, flat);
            if (total > 0)
            {
                constexpr bool kOdd   = INTERP == NVCV_INTERP_CUBIC && kFixedCubic<T> && C != 4;
                auto           kernel = kOdd && RowsAreOdd<C>(srcHost + first, count) ? ResizePatchVarShapeKernel<T, C, INTERP, kOdd>
                                                                                      : ResizePatchVarShapeKernel<T, C, INTERP, false>;
                hipLaunchKernelGGL(kernel, dim3(total), dim3(256), 0, stream, a,
                                   tiles, (int)flat);
                CheckLaunch("ResizePatchVarShapeKernel");
            }
            continue;
        }
        int total = BuildVarTiles(tiles, dstHost, first, count, kTileW, kTileH);
        if (total > 0)
        {
            hipLaunchKernelGGL((ResizeVarShapeKernel<T, C, INTERP>), dim3(total), dim3(256), 0, stream, a, tiles);
            CheckLaunch("ResizeVarShapeKernel");
        }
    }
}

template<class T, int C>
void DispatchInterp(bool varshape, const ResizeArgs &a, const NVCVImageBufferStrided *srcHost,
                    const NVCVImageBufferStrided *dstHost, int N, int interp,
                    hipStream_t stream)
{
    switch (interp)
    {
    case NVCV_INTERP_NEAREST:
        varshape ? LaunchVarShape<T, C, NVCV_INTERP_NEAREST>(a, srcHost, dstHost, N, stream)
                 : LaunchTensor<T, C, NVCV_INTERP_NEAREST>(a, N, stream);
        break;
    case NVCV_INTERP_LINEAR:
        varshape ? LaunchVarShape<T, C, NVCV_INTERP_LINEAR>(a, srcHost, dstHost, N, stream)
                 : LaunchTensor<T, C, NVCV_INTERP_LINEAR>(a, N, stream);
        break;
    case NVCV_INTERP_CUBIC:
        varshape ? LaunchVarShape<T, C, NVCV_INTERP_CUBIC>(a, srcHost, dstHost, N, stream)
                 : LaunchTensor<T, C, NVCV_INTERP_CUBIC>(a, N, stream);
        break;
    case NVCV_INTERP_AREA:
        varshape ? LaunchVarShape<T, C, NVCV_INTERP_AREA>(a, srcHost, dstHost, N, stream)
                 : LaunchTensor<T, C, NVCV_INTERP_AREA>(a, N, stream);
        break;
    default:
        throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Invalid interpolation (supported: NEAREST, LINEAR, CUBIC, AREA)");
    }
}

template<class T>
void DispatchChannels(int channels, bool varshape, const ResizeArgs &a, const NVCVImageBufferStrided *srcHost,
                      const NVCVImageBufferStrided *dstHost, int N,
                      int interp, hipStream_t stream)
{
    switch (channels)
    {
    case 1:
        DispatchInterp<T, 1>(varshape, a, srcHost, dstHost, N, interp, stream);
        break;
    case 3:
        DispatchInterp<T, 3>(varshape, a, srcHost, dstHost, N, interp, stream);
        break;
    case 4:
        DispatchInterp<T, 4>(varshape, a, srcHost, dstHost, N, interp, stream);
        break;
    default:
        throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Invalid input data type");
    }
}

void DispatchType(ElemType elem, int channels, bool varshape, const ResizeArgs &a, const NVCVImageBufferStrided *srcHost,
                  const NVCVImageBufferStrided *dstHost, int N, int interp, hipStream_t stream)
{
    if (N == 0)
    {
        return;
    }
    switch (elem)
    {
    case kU8:
        DispatchChannels<uint8_t>(channels, varshape, a, srcHost, dstHost, N, interp, stream);
        break;
    case kU16:
        DispatchChannels<uint16_t>(channels, varshape, a, srcHost, dstHost, N, interp, stream);
        break;
    case kS16:
        DispatchChannels<int16_t>(channels, varshape, a, srcHost, dstHost, N, interp, stream);
        break;
    case kF32:
        DispatchChannels<float>(channels, varshape, a, srcHost, dstHost, N, interp, stream);
        break;
    default:
        throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Invalid input data type");
    }
}

class Resize final : public IOperator
{
public:
    void submit(hipStream_t stream, NVCVTensorHandle hin, NVCVTensorHandle hout, NVCVInterpolationType interp) const
    {
        NVCVTensorData din, dout;
        ExportTensor(hin, din, "Input");
        ExportTensor(hout, dout, "Output");
        if (din.dtype != dout.dtype)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Input and output data type are different");
        }
        if (nvcvTensorLayoutCompare(din.layout, dout.layout) != 0)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Input and output data layout are different");
        }
        if (nvcvTensorLayoutCompare(din.layout, NVCV_TENSOR_HWC) != 0
            && nvcvTensorLayoutCompare(din.layout, NVCV_TENSOR_NHWC) != 0)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Input must have (N)HWC layout");
        }
        ImageBatchView in  = RequireImageBatchView(din, "Input", NVCV_ERROR_INVALID_ARGUMENT);
        ImageBatchView out = RequireImageBatchView(dout, "Output", NVCV_ERROR_INVALID_ARGUMENT);
        if (in.N != out.N)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Input and output samples are different");
        }
        if (in.C != out.C)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Input and output channels are different");
        }
        if (in.C > 4 || in.C < 1)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Invalid number of channels");
        }
        if (std::max(in.bytesSpanned(), out.bytesSpanned()) > INT32_MAX)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Input or output tensors are too large");
        }
        ResizeArgs a      = {};
        a.srcBase         = in.base;
        a.dstBase         = out.base;
        a.srcSampleStride = in.strideN;
        a.dstSampleStride = out.strideN;
        a.srcRowStride    = (int32_t)in.strideH;
        a.dstRowStride    = (int32_t)out.strideH;
        a.srcW            = in.W;
        a.srcH            = in.H;
        a.dstW            = out.W;
        a.dstH            = out.H;
        if (out.W == 0 || out.H == 0)
        {
            return;
        }
        a.scaleX = static_cast<float>(in.W) / out.W; // IEEE float32 division, as the kernels would do it
        a.scaleY = static_cast<float>(in.H) / out.H;
        DispatchType(in.elem, in.C, false, a, nullptr, nullptr, in.N, interp, stream);
    }

    void submit(hipStream_t stream, NVCVImageBatchHandle hin, NVCVImageBatchHandle hout,
                NVCVInterpolationType interp) const
    {
        VarShapeView in  = ExportVarShape(hin, stream, "Input");
        VarShapeView out = ExportVarShape(hout, stream, "Output");
        if (in.N != out.N)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Invalid input and output batch sizes: %d != %d", in.N, out.N);
        }
        if (in.uniqueFormat == NVCV_IMAGE_FORMAT_NONE || in.uniqueFormat != out.uniqueFormat)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT,
                          "All images in the input and output batches must share one format");
        }
        FormatInfo fi = DecodeFormat(in.uniqueFormat);
        if (fi.planes != 1)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Images must have a single interleaved plane");
        }
        ResizeArgs a = {};
        a.srcList    = in.data.buffer.varShapeStrided.imageList;
        a.dstList    = out.data.buffer.varShapeStrided.imageList;
        DispatchType(fi.elem, fi.channels, true, a, in.hostList, out.hostList, in.N, interp, stream);
    }
};

} // namespace
} // namespace cvamd

using namespace cvamd;

extern "C"
{
CVCUDA_PUBLIC NVCVStatus cvcudaResizeCreate(NVCVOperatorHandle *handle)
{
    return CreateOperator<Resize>(handle);
}

CVCUDA_PUBLIC NVCVStatus cvcudaResizeSubmit(NVCVOperatorHandle handle, hipStream_t stream, NVCVTensorHandle in,
                                            NVCVTensorHandle out, const NVCVInterpolationType interpolation)
{
    return Protect([&] { ToOperator<Resize>(handle).submit(stream, in, out, interpolation); });
}

CVCUDA_PUBLIC NVCVStatus cvcudaResizeVarShapeSubmit(NVCVOperatorHandle handle, hipStream_t stream,
                                                    NVCVImageBatchHandle in, NVCVImageBatchHandle out,
                                                    const NVCVInterpolationType interpolation)
{
    return Protect([&] { ToOperator<Resize>(handle).submit(stream, in, out, interpolation); });
}
}

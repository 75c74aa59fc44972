// WarpAffine and WarpPerspective, tensors and var-shape batches.
//
// Coordinates, sampling and border handling follow the reference in float32 without FMA
// contraction (the bilinear sum in the association of the reference's golden, tap * (wx * wy),
// tests/cvcuda/system/TestOpWarpAffine.cpp:159-170, so integer results equal the golden's bit for bit; bicubic weights and sums
// of floats and of 8-bit pixels are the exceptions, see CubicWeights and kFixedPointCubic): destination->source map src/cvcuda/priv/legacy/CvCudaLegacy.h:143-183, matrix
// inversion warp.cu:139-150 (affine) and cuda_tools/math/LinAlg.hpp:1446-1450, 1640-1654 (3x3),
// samplers cuda_tools/InterpolationWrap.hpp:83-104, 332-339, 429-447, 535-565, border index maps
// cuda_tools/BorderWrap.hpp:62-121. Validation follows warp.cu:152-232 and warp_var_shape.cu:194-299.
//
// Differences by design: the var-shape kernels read each image's matrix straight from the caller's
// [N,6] / [N,9] tensor and invert it in the block prologue (a few scalar operations), so the operator
// owns no device buffer and launches no separate inversion kernel; several var-shape submissions of
// one operator handle may therefore be in flight at once. Var-shape batches run on a packed tile grid.
//
// Kernel shape. A 256-thread block produces a 64 x 16 pixel tile of the destination (64 x 8 in small launches); each of its four
// waves works on its own 32 x 8 (16 x 8) part, no barrier.
// Gather: the cost of the gather is set by how many distinct cache lines one wave-wide load touches,
// and under a rotation every source row a wave's footprint crosses is another line; so a wave samples
// compact 8 x 8 pixel patches (one lane per pixel, ~10 source rows per load where a 64 x 1 strip would
// cross ~20), four patches (two) side by side per wave, i.e. 4 (2) independent samples per lane
// whose loads are in flight together. Taps that lie inside the source image - nearly all of them -
// skip the border logic and fetch the horizontally adjacent taps of a row with one load (u8x3: the 6
// bytes of two pixels from an aligned 12-byte window).
// Store: "one pixel in each patch" becomes "4 consecutive pixels of one row" through LDS, which the lane writes as whole
// dwords; single-byte stores scattered over 8 rows are several times slower. Pixels of 12 and 16 bytes leave as whole rows of the wave's part, 16 bytes per lane.
#include "DeviceUtils.hpp"
#include "FixedPointBlend.hpp"
#include "LaneExchange.hpp"
#include "OpCommon.hpp"
#include "VarShapeTiles.hpp"

#include <cvcuda/OpWarpAffine.h>
#include <cvcuda/OpWarpPerspective.h>

#include <algorithm>
#include <cmath>

namespace cvamd {

namespace {

constexpr int kPatch   = 8; // gather granule: a wave samples kPatch x kPatch pixels per step
// A wave's N patches lie side by side, N = kMostPatches or kFewPatches (see LaunchMap); a block's waves as two by two, four in a
// row or one alone.
constexpr int kMostPatches = 4, kFewPatches = 2;
template<int N>
constexpr int kWaveW = kPatch * N;

// A block of 64 x WAVES threads.
template<int N, int WAVES>
struct Block
{
    static constexpr int kWaves = WAVES, kThreads = 64 * WAVES;
    static constexpr int kAcross = WAVES == 1 ? 1 : N == kMostPatches ? 2 : 4;
    static constexpr int kTileW = kWaveW<N> * kAcross, kTileH = WAVES / kAcross * kPatch;
};

// Waves of 8-bit bicubic with three channels are the longest and their lengths differ most (the image's edge), so a block of four holds its
// places until the last one ends: in large launches, and where blocks of four have waves outside the images, they go alone. us with four
// waves / one: 24 images of 697 .. 1194 x 187 .. 545 39.0 / 36.2, 9 x 1241 x 955 in perspective 48.1 / 46.8. Others gain nothing by it (u8x4 34.6 /
// 35.0, u8x1 41.0 / 41.1) or are held up by the launch of so many blocks, 4.6 a ns at most (nearest neighbour u8x1 27.2 / 36.2, u8x3 85.9 /
// 102.5, bilinear u8x3 48.1 / 53.4).
template<class T, int C, int INTERP, int N>
constexpr bool kSingleWaves = std::is_same_v<T, uint8_t> && C == 3 && INTERP == NVCV_INTERP_CUBIC && N == kMostPatches;

// The waves of a launch in blocks of one and, with those that stand outside the images, of four. Time of one over four in 400 random launches, inputs
// and outputs out of the memory's cache: none outside and up to 32 768 waves 1.01 to 1.03 (160 x 196 x 29 11.0 us / 13.6), beyond 0.99 and
// 0.94; 2 % to 10 % outside and up to 8192 waves 1.00 to 1.05, beyond 0.89 to 0.99; 10 % to 20 % 0.97 to 1.00 and 0.87 to 0.91; more 0.63 to 0.97.
constexpr bool SingleWavesPay(int64_t ones, int64_t fours)
{
    return ones > 32768 || 10 * fours >= 11 * ones || (ones > 8192 && 50 * fours >= 51 * ones);
}

struct WarpArgs
{
    const uint8_t *src;
    uint8_t       *dst;
    int64_t        srcN, dstN;
    int32_t        srcRow, dstRow;
    int32_t        srcW, srcH, dstW, dstH;
    const NVCVImageBufferStrided *srcList;
    const NVCVImageBufferStrided *dstList;
    // matrix: tensor path -> m[] already maps dst->src; var-shape -> rows of `xforms`
    float          m[9];
    const uint8_t *xforms;
    int64_t        xformStride; // bytes between matrices
    int32_t        inverseGiven; // var-shape: 1 = matrices already map dst->src
    int32_t        perspective;
    int32_t        border;
    float          bval[4];
};

template<class T, int C>
using Vec = Packed<T, C>;

struct Img
{
    const uint8_t *base;
    int32_t        row, w, h;
};

template<class T, int C>
__device__ __forceinline__ void Fetch(const Img &im, const WarpArgs &a, int x, int y, float (&out)[C])
{
    if (a.border == NVCV_BORDER_CONSTANT)
    {
        if (x < 0 || x >= im.w || y < 0 || y >= im.h)
        {
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                out[c] = (float)BorderValueAs<T>(a.bval[c]);
            }
            return;
        }
    }
    else
    {
        x = BorderIndex(a.border, x, im.w);
        y = BorderIndex(a.border, y, im.h);
    }
    const Vec<T, C> px = reinterpret_cast<const Vec<T, C> *>(im.base + (int64_t)y * im.row)[x];
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        out[c] = (float)px.v[c];
    }
}

__device__ __forceinline__ void CubicCoeffs(float d, float (&w)[4])
{
    w[0] = -.5f;
    w[0] = w[0] * d + 1.f;
    w[0] = w[0] * d - .5f;
    w[0] = w[0] * d;
    w[1] = 1.5f;
    w[1] = w[1] * d - 2.5f;
    w[1] = w[1] * d;
    w[1] = w[1] * d + 1.f;
    w[2] = -1.5f;
    w[2] = w[2] * d + 2.f;
    w[2] = w[2] * d + .5f;
    w[2] = w[2] * d;
    w[3] = 1 - w[0] - w[1] - w[2];
}

// float -> int index like the reference's round-down conversion; huge / non-finite coordinates
// saturate instead of invoking undefined behaviour
__device__ __forceinline__ int FloorToInt(float v)
{
    return (int)fminf(fmaxf(floorf(v), -1073741824.f), 1073741824.f);
}

// 8-bit bilinear: the blend of FixedPointBlend.hpp; the fractions are ax = trunc(fx * 2^15) with
// fx = sx - floor(sx) in float32. Integer and quarter-step maps (the reference's own exact-equality table)
// give weights that are exact in both arithmetics, hence the same results as the reference's golden.
template<class T, int INTERP>
constexpr bool kFixedPoint = std::is_same_v<T, uint8_t> && INTERP == NVCV_INTERP_LINEAR;

// 8-bit bicubic: the four horizontal weights (the reference's float32 polynomials) are rounded to
// multiples of 2^-14 with the last one taking the remainder, so that they add up to exactly 1; a row's
// four taps are combined in integers (exact), the four row sums in float32 with the vertical weights.
// Every horizontal weight is within 2^-15 of the float32 one (the last within 2^-14): the result is
// within 0.05 of the float32 expression's, i.e. at most 1 from the reference's golden.
template<class T, int INTERP>
constexpr bool kFixedPointCubic = std::is_same_v<T, uint8_t> && INTERP == NVCV_INTERP_CUBIC;

// The kernels that blend in fixed point work on coordinates in units of 2^-15 pixel: the first two rows
// of their destination -> source matrix arrive multiplied by 2^15 (exact: a power of two), so floor and
// fraction of a coordinate are the two halves of one float -> integer conversion.
template<class T, int INTERP>
constexpr float kCoordScale = kFixedPoint<T, INTERP> ? 32768.f : 1.f;

// floor and 15-bit fraction of a coordinate; NaN and infinite coordinates give fraction 0
__device__ __forceinline__ uint32_t FractionQ15(float v)
{
    const float f = v - floorf(v);
    return f >= 0.f ? (uint32_t)(int)(f * 32768.f) : 0u;
}

// CubicCoeffs times `scale` (a power of two, so every step scales exactly) with the polynomials evaluated
// by fused multiply-adds; used where the weights are quantised afterwards anyway.
__device__ __forceinline__ void CubicCoeffsFused(float d, float scale, float (&w)[4])
{
    w[0] = __builtin_fmaf(-.5f * scale, d, scale);
    w[0] = __builtin_fmaf(w[0], d, -.5f * scale);
    w[0] = w[0] * d;
    w[1] = __builtin_fmaf(1.5f * scale, d, -2.5f * scale);
    w[1] = w[1] * d;
    w[1] = __builtin_fmaf(w[1], d, scale);
    w[2] = __builtin_fmaf(-1.5f * scale, d, 2.f * scale);
    w[2] = __builtin_fmaf(w[2], d, .5f * scale);
    w[2] = w[2] * d;
    w[3] = scale - w[0] - w[1] - w[2];
}

// The bicubic weights and sums of other than 8-bit pixels: the reference's products tap * (wx * wy) in its order; of floats by
// fused multiply-adds, 32 vector instructions of a pixel for 48, whose sums are rounded half as often: against 64-bit sums over
// the same places they differ by 0.92e-7 of the norm where separate ones did by 0.97e-7 (three channels about zero 1.1e-7 and
// 1.25e-7). With a row's taps in one load 17 x 915 x 2004 f32x1 180 -> 120 us (its L1 accesses, 24 per load, had been all of
// the launch), 16 x 2048 x 315 f32x3 114 -> 95.
template<class T>
__device__ __forceinline__ void CubicWeights(float d, float (&w)[4])
{
    if constexpr (std::is_same_v<T, float>)
    {
        CubicCoeffsFused(d, 1.f, w);
    }
    else
    {
        CubicCoeffs(d, w);
    }
}

template<class T, int INTERP>
__device__ __forceinline__ float AddTap(float acc, float tap, float weight)
{
    return std::is_same_v<T, float> && INTERP == NVCV_INTERP_CUBIC ? __builtin_fmaf(tap, weight, acc) : acc + tap * weight;
}

// Taps of 1 and 3 bytes are fetched through dword-aligned windows, as many dwords as hold the taps of a row wherever they
// start (single bytes as they are). Windows read up to 2 pixels (u8x3) past the taps, 6 (u8x1 bilinear) or 4 (bicubic):
// harmless inside the image; taps that close to the end of a row, and so of the image, are kept off this path by TapsInside.
template<class T, int C>
constexpr bool kWideTapLoads = std::is_same_v<T, uint8_t> && (C == 1 || C == 3);

template<class T, int C, int INTERP>
constexpr int kTapOverrun = !kWideTapLoads<T, C>          ? 0
                          : C == 3                        ? 2
                          : INTERP == NVCV_INTERP_NEAREST ? 0
                          : INTERP == NVCV_INTERP_LINEAR  ? 6
                                                          : 4;

// One pixel at base + off, known to be inside the image.
template<class T, int C>
__device__ __forceinline__ void LoadPixelInside(const uint8_t *base, uint32_t off, T (&out)[C])
{
    const Vec<T, C> v = *reinterpret_cast<const Vec<T, C> *>(base + off);
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        out[c] = v.v[c];
    }
}

// Two horizontally adjacent pixels starting at base + off, both known to be inside the image.
template<class T, int C>
__device__ __forceinline__ void LoadPairInside(const uint8_t *base, uint32_t off, float (&p0)[C], float (&p1)[C])
{
    const Vec<T, 2 * C> v = *reinterpret_cast<const Vec<T, 2 * C> *>(base + off);
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        p0[c] = (float)v.v[c];
        p1[c] = (float)v.v[C + c];
    }
}

// Byte offset of pixel (x, y), both inside the image. Image planes are below 2 GiB. Uses the 24-bit
// multiply (full rate; the 32-bit one runs at a quarter): images whose row pitch or height does not
// fit 23 bits never take the path that calls this.
template<int PIXEL_BYTES>
__device__ __forceinline__ uint32_t PixelOffset(const Img &im, int x, int y)
{
    return (uint32_t)__mul24(y, im.row) + (uint32_t)x * PIXEL_BYTES;
}

// 1 / x, correctly rounded, for 2^-123 <= |x| < 2^123: the hardware's approximation (within one unit in the last place) and
// one correction by the residual, which fused multiply-adds form and apply without rounding in between (P. Markstein,
// Computation of elementary functions on the IBM RISC System/6000 processor, 1990). Equal to the quotient for all 2^23
// mantissas of both signs at every exponent in the range on gfx950.
__device__ __forceinline__ float ReciprocalInRange(float x)
{
    const float r = __builtin_amdgcn_rcpf(x);
    return __builtin_fmaf(__builtin_fmaf(-x, r, 1.f), r, r);
}

// The source coordinates of a lane's samples at the destination pixels (dx[k], dy[k]), as MapCoord gives them. A perspective's
// quotients are 3 instructions instead of 10 where all of them are in ReciprocalInRange's range (16 x 1240 x 1754 u8x3
// bicubic: see BlendCubicQ14).
template<bool PERSPECTIVE, int N>
__device__ __forceinline__ void MapCoords(const float (&m)[9], const int (&dx)[N], const int (&dy)[N], float (&sx)[N], float (&sy)[N])
{
    if constexpr (PERSPECTIVE)
    {
        float    coeff[N];
        uint32_t low = 0xffffffffu, high = 0;
#pragma unroll
        for (int k = 0; k < N; ++k)
        {
            coeff[k] = m[6] * dx[k] + m[7] * dy[k] + m[8];
            low      = min(low, __float_as_uint(coeff[k]) & 0x7fffffffu);
            high     = max(high, __float_as_uint(coeff[k]) & 0x7fffffffu);
        }
        if (low >= (4u << 23) && high < (250u << 23))
        {
#pragma unroll
            for (int k = 0; k < N; ++k)
            {
                coeff[k] = ReciprocalInRange(coeff[k]);
            }
        }
        else
        {
#pragma nounroll
            for (int k = 0; k < N; ++k)
            {
                float c = coeff[0];
#pragma unroll
                for (int j = 1; j < N; ++j)
                {
                    c = j == k ? coeff[j] : c;
                }
                const float q = 1.0f / c;
#pragma unroll
                for (int j = 0; j < N; ++j)
                {
                    coeff[j] = j == k ? q : coeff[j];
                }
            }
        }
#pragma unroll
        for (int k = 0; k < N; ++k)
        {
            sx[k] = coeff[k] * (m[0] * dx[k] + m[1] * dy[k] + m[2]);
            sy[k] = coeff[k] * (m[3] * dx[k] + m[4] * dy[k] + m[5]);
        }
    }
    else
    {
#pragma unroll
        for (int k = 0; k < N; ++k)
        {
            sx[k] = m[0] * dx[k] + m[1] * dy[k] + m[2];
            sy[k] = m[3] * dx[k] + m[4] * dy[k] + m[5];
        }
    }
}

template<bool PERSPECTIVE>
__device__ __forceinline__ void MapCoord(const float (&m)[9], int dx, int dy, float &sx, float &sy)
{
    if constexpr (PERSPECTIVE)
    {
        const float coeff = 1.0f / (m[6] * dx + m[7] * dy + m[8]);
        sx                = coeff * (m[0] * dx + m[1] * dy + m[2]);
        sy                = coeff * (m[3] * dx + m[4] * dy + m[5]);
    }
    else
    {
        sx = m[0] * dx + m[1] * dy + m[2];
        sy = m[3] * dx + m[4] * dy + m[5];
    }
}

// One destination pixel sampled at (sx, sy) with every tap going through the border logic. The tap
// loops are deliberately not unrolled: this path runs only for the few waves that straddle the image
// border, and one copy of the border code keeps the kernel small.
template<class T, int C, int INTERP>
__device__ __forceinline__ void SampleWithBorder(const Img &im, const WarpArgs &a, float sx, float sy, T (&out)[C])
{
    float acc[C];
    if constexpr (INTERP == NVCV_INTERP_NEAREST)
    {
        Fetch<T, C>(im, a, FloorToInt(sx + .5f), FloorToInt(sy + .5f), acc);
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            out[c] = (T)acc[c]; // the tap itself (exactly representable), no rounding involved
        }
        return;
    }
    else if constexpr (kFixedPoint<T, INTERP>)
    {
        const int      x1 = FloorToInt(sx), y1 = FloorToInt(sy);
        const uint32_t ax = FractionQ15(sx), ay = FractionQ15(sy);
        const uint32_t w11 = (ax * ay + (kQ15 >> 1)) >> 15;
        uint32_t       sum[C];
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            sum[c] = 0;
        }
#pragma nounroll
        for (int i = 0; i < 4; ++i) // taps (x1,y1) (x2,y1) (x1,y2) (x2,y2)
        {
            float t[C];
            Fetch<T, C>(im, a, x1 + (i & 1), y1 + (i >> 1), t);
            const uint32_t w = i == 0 ? kQ15 - ax - ay + w11 : (i == 1 ? ax - w11 : (i == 2 ? ay - w11 : w11));
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                sum[c] += (uint32_t)t[c] * w;
            }
        }
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            out[c] = RoundQ15(sum[c]);
        }
        return;
    }
    else if constexpr (INTERP == NVCV_INTERP_LINEAR)
    {
        const int x1 = FloorToInt(sx), y1 = FloorToInt(sy);
        const int x2 = x1 + 1, y2 = y1 + 1;
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            acc[c] = 0.f;
        }
#pragma nounroll
        for (int i = 0; i < 4; ++i) // taps (x1,y1) (x2,y1) (x1,y2) (x2,y2) in this order
        {
            float t[C];
            Fetch<T, C>(im, a, x1 + (i & 1), y1 + (i >> 1), t);
            const float wx = (i & 1) ? (sx - x1) : (x2 - sx);
            const float wy = (i >> 1) ? (sy - y1) : (y2 - sy);
            const float w  = wx * wy;
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                acc[c] += t[c] * w;
            }
        }
    }
    else if constexpr (kFixedPointCubic<T, INTERP>)
    {
        const int ix = FloorToInt(sx), iy = FloorToInt(sy);
        float     wx[4], wy[4];
        CubicCoeffsFused(sx - floorf(sx), 16384.f, wx);
        CubicCoeffsFused(sy - floorf(sy), 1.f / 16384.f, wy);
        int wq[4];
        CubicWeightsQ14(wx, wq);
#pragma nounroll
        for (int cy = 0; cy < 4; ++cy)
        {
            int h[C];
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                h[c] = 0;
            }
#pragma nounroll
            for (int cx = 0; cx < 4; ++cx)
            {
                float t[C];
                Fetch<T, C>(im, a, ix + cx - 1, iy + cy - 1, t);
                const int w = cx == 0 ? wq[0] : (cx == 1 ? wq[1] : (cx == 2 ? wq[2] : wq[3]));
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    h[c] += (int)t[c] * w;
                }
            }
            const float v = cy == 0 ? wy[0] : (cy == 1 ? wy[1] : (cy == 2 ? wy[2] : wy[3]));
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                acc[c] = cy == 0 ? (float)h[c] * v : __builtin_fmaf((float)h[c], v, acc[c]);
            }
        }
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            out[c] = SaturateCast<T>(acc[c]);
        }
        return;
    }
    else
    {
        const int ix = FloorToInt(sx), iy = FloorToInt(sy);
        float     wx[4], wy[4];
        CubicWeights<T>(sx - ix, wx);
        CubicWeights<T>(sy - iy, wy);
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            acc[c] = 0.f;
        }
#pragma unroll
        for (int cy = 0; cy < 4; ++cy)
        {
#pragma unroll
            for (int cx = 0; cx < 4; ++cx)
            {
                float t[C];
                Fetch<T, C>(im, a, ix + cx - 1, iy + cy - 1, t);
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    acc[c] = AddTap<T, INTERP>(acc[c], t[c], wx[cx] * wy[cy]);
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        out[c] = SaturateCast<T>(acc[c]);
    }
}

// True when every tap of the sample at (sx, sy) lies inside the image (and none of them is among
// the image's last kTapOverrun columns: the window loads read that far past a row's taps, which must not run off the end
// of the last row). limX / limY come from InsideLimits. For an integer k,
// floor(v) < k <=> v < k, so the test is 0 <= v - lo < lim per axis, done as ONE unsigned comparison
// of the float's bit pattern: non-negative floats order like their bits, negative ones and NaNs have
// patterns above every finite positive limit (-0.0 fails too and takes the generic path, which
// computes the same result).
// The test runs on a lane's N samples at once: the largest bit pattern per axis against the limit.
template<int INTERP, int N>
__device__ __forceinline__ bool TapsInside(float limX, float limY, const float (&sx)[N], const float (&sy)[N])
{
    // taps span [floor(v) - lo, floor(v) + hi] per axis; NEAREST takes floor(v + .5)
    constexpr float lo = INTERP == NVCV_INTERP_CUBIC ? 1.f : (INTERP == NVCV_INTERP_NEAREST ? -.5f : 0.f);
    uint32_t        ux = 0, uy = 0;
#pragma unroll
    for (int k = 0; k < N; ++k)
    {
        ux = max(ux, __float_as_uint(sx[k] - lo));
        uy = max(uy, __float_as_uint(sy[k] - lo));
    }
    return (ux < __float_as_uint(limX)) & (uy < __float_as_uint(limY)); // bitwise on purpose: no branch
}

template<int INTERP>
__device__ __forceinline__ bool TapInside(float limX, float limY, float sx, float sy)
{
    constexpr float lo = INTERP == NVCV_INTERP_CUBIC ? 1.f : (INTERP == NVCV_INTERP_NEAREST ? -.5f : 0.f);
    return (__float_as_uint(sx - lo) < __float_as_uint(limX)) & (__float_as_uint(sy - lo) < __float_as_uint(limY));
}

// Exclusive upper limit of floor(v) - lo along an axis of `size` pixels; 0 (no sample passes) when the
// image is smaller than the tap span.
template<int INTERP>
__device__ __forceinline__ float InsideLimit(int size, int overrun)
{
    constexpr int lo = INTERP == NVCV_INTERP_CUBIC ? 1 : 0;
    constexpr int hi = INTERP == NVCV_INTERP_CUBIC ? 2 : (INTERP == NVCV_INTERP_LINEAR ? 1 : 0);
    return (float)max(size - hi - lo - overrun, 0);
}

// Same arithmetic as SampleWithBorder for a sample whose taps are all inside the image: no border
// logic, adjacent taps fetched together, no branches (so the loads of several pixels can be in flight
// at once). floorf(v) is used directly where the generic path converts floor(v) to int and back.
// O = T, or float for the unrounded sums (not for NEAREST).
template<class O, int C, int INTERP, class T = O>
__device__ __forceinline__ void SampleInside(const Img &im, float sx, float sy, O (&out)[C])
{
    constexpr int PB = C * sizeof(T);
    float         acc[C];
    if constexpr (INTERP == NVCV_INTERP_NEAREST)
    {
        const int x = (int)floorf(sx + .5f), y = (int)floorf(sy + .5f);
        LoadPixelInside<T, C>(im.base, PixelOffset<PB>(im, x, y), out);
        return;
    }
    else if constexpr (INTERP == NVCV_INTERP_LINEAR)
    {
        const float fx = floorf(sx), fy = floorf(sy);
        const float wx1 = sx - fx, wx0 = (fx + 1.f) - sx;
        const float wy1 = sy - fy, wy0 = (fy + 1.f) - sy;
        const uint32_t o = PixelOffset<PB>(im, (int)fx, (int)fy);
        float          t[4][C];
        LoadPairInside<T, C>(im.base, o, t[0], t[1]);
        LoadPairInside<T, C>(im.base, o + (uint32_t)im.row, t[2], t[3]);
        const float w00 = wx0 * wy0, w01 = wx1 * wy0, w10 = wx0 * wy1, w11 = wx1 * wy1;
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            float v = t[0][c] * w00;
            v += t[1][c] * w01;
            v += t[2][c] * w10;
            v += t[3][c] * w11;
            acc[c] = v;
        }
    }
    else
    {
        const float fx = floorf(sx), fy = floorf(sy);
        float       wx[4], wy[4];
        CubicWeights<T>(sx - fx, wx);
        CubicWeights<T>(sy - fy, wy);
        uint32_t o = PixelOffset<PB>(im, (int)fx - 1, (int)fy - 1);
        float    t[4][4][C];
#pragma unroll
        for (int cy = 0; cy < 4; ++cy)
        {
            // (4 pixels at once: pairs of f32x1 were twice as many loads, of f32x3 four for these three)
            const Vec<T, 4 * C> v = *reinterpret_cast<const Vec<T, 4 * C> *>(im.base + o);
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    t[cy][i][c] = (float)v.v[i * C + c];
                }
            }
            o += (uint32_t)im.row;
        }
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            acc[c] = 0.f;
        }
#pragma unroll
        for (int cy = 0; cy < 4; ++cy)
        {
#pragma unroll
            for (int cx = 0; cx < 4; ++cx)
            {
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    acc[c] = AddTap<T, INTERP>(acc[c], t[cy][cx][c], wx[cx] * wy[cy]);
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        if constexpr (std::is_same_v<O, T>)
        {
            out[c] = SaturateCast<T>(acc[c]);
        }
        else
        {
            out[c] = acc[c];
        }
    }
}

// A uniform address that stays one: without this the compiler adds the row's part to each lane's 64-bit address.
__device__ __forceinline__ const uint8_t *UniformRow(const uint8_t *row)
{
    uintptr_t at = reinterpret_cast<uintptr_t>(row);
    asm("" : "+s"(at));
    return AsGlobal(reinterpret_cast<const uint8_t *>(at));
}

// How the taps of a row are read: windows whose rows' addresses differ in their low two bits, or agree in them (a row pitch
// of whole dwords); or a load of the taps alone at any address (single-channel pixels, see NarrowTapsPay).
enum RowForm
{
    kOddRows,
    kSameRows,
    kNarrowTaps
};

// The rows y .. y + ROWS - 1 of a u8 image, from pixel x on (TAPS pixels, all inside the image), as raw bytes: r[j] holds row
// j's. Per sample this is two multiply-adds for the offset, whose start (uniform) takes in what is added to x and y, and, where
// the rows' addresses agree in their low two bits, one mask: a row's address is its own
// uniform base plus that one offset. Written with the compiler's choice of instructions and the row pitch added per lane,
// the kernel had a fifth more vector instructions (bilinear; bicubic a ninth). Single-channel taps, which had been fetched as
// 2- and 4-byte loads at any address, gain most, by the loads: one that is not dword aligned is taken apart (a gather of
// u8x3 pixel pairs: 31 against 22 cycles per wave). 24 x 1283 x 721 u8x1 bilinear 54.3 -> 43.0 us, bicubic 131.3 -> 100.7;
// 16 x 1280 x 720 u8x3 bicubic 68.4 -> 64.6, bilinear 30.1 -> 29.2 (which the L1 accesses of its gathers
// bound now: 54 us of the 63 that 32 x 1280 x 780 take, against 45 of issue).
template<int C, int TAPS, int ROWS, int FORM>
__device__ __forceinline__ void LoadTapRows(const Img &im, int x, int y, int x0, int y0, uint32_t (&r)[ROWS][(C * TAPS + 3) / 4])
{
    constexpr int  N       = (C * TAPS + 3) / 4;
    constexpr bool kWindow = kWideTapLoads<uint8_t, C> && C * TAPS > 1 && FORM != kNarrowTaps, SAME = FORM == kSameRows;
    constexpr int  kLoad   = kWindow ? (C * TAPS + 3 + 3) / 4 : N; // dwords that hold C * TAPS bytes at any of the 4 places
    struct alignas(4) W
    {
        uint32_t d[kLoad];
    };
    const uint32_t mis0  = kWindow ? (uint32_t)reinterpret_cast<uintptr_t>(im.base) & 3u : 0u;
    const int      start = y0 * im.row + x0 * C + (int)mis0;
    uint32_t       o;
    asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(o) : "v"(x), "n"(C), "s"(start));
    asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(o) : "v"(y), "s"(im.row), "v"(o));
    W w[ROWS];
    if constexpr (kWindow)
    {
        uint32_t       shift[ROWS];
        const uint8_t *base = im.base - mis0;
#pragma unroll
        for (int j = 0; j < ROWS; ++j)
        {
            // (in a row pitch that is not of whole dwords, row j's base starts at a dword and its offset grows by the rest)
            const uint32_t rest = SAME ? 0u : (mis0 + (uint32_t)(j * im.row)) & 3u;
            shift[j]            = SAME ? o : o - mis0 + rest;
            const uint8_t *row  = UniformRow(SAME ? base + j * im.row : im.base + j * im.row - rest);
            w[j]                = *reinterpret_cast<const W *>(row + (shift[j] & ~3u));
        }
#pragma unroll
        for (int j = 0; j < ROWS; ++j)
        {
#pragma unroll
            for (int i = 0; i < N; ++i)
            {
                r[j][i] = __builtin_amdgcn_alignbyte(i + 1 < kLoad ? w[j].d[i + 1] : w[j].d[i], w[j].d[i], shift[j]);
            }
        }
    }
    else
    {
#pragma unroll
        for (int j = 0; j < ROWS; ++j)
        {
            const Vec<uint8_t, C * TAPS> v = *reinterpret_cast<const Vec<uint8_t, C * TAPS> *>(UniformRow(im.base + j * im.row) + o);
            r[j][N - 1]                    = 0;
            __builtin_memcpy(r[j], &v, C * TAPS);
        }
    }
}

// The fixed-point bicubic sum (see kFixedPointCubic) of the 4 x 4 taps in r (row j, 4 pixels as raw bytes).
template<int C>
__device__ __forceinline__ uint32_t BlendCubicQ14(const uint32_t (&r)[4][C], float sx, float sy)
{
    float wx[4], wy[4];
    CubicCoeffsFused(sx - floorf(sx), 16384.f, wx);
    CubicCoeffsFused(sy - floorf(sy), 1.f / 16384.f, wy);
    uint32_t p01, p23;
    CubicWeightPairsQ14(wx, p01, p23);
    uint32_t q = 0;
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            const float h = RowSumQ14(BytePair(r[j], c, c + C), BytePair(r[j], c + 2 * C, c + 3 * C), p01, p23);
            acc           = j == 0 ? h * wy[0] : __builtin_fmaf(h, wy[j], acc);
        }
        q = __builtin_amdgcn_cvt_pk_u8_f32(acc, c, q);
    }
    return q;
}

// The same for a sample whose 16 taps are inside the image.
template<int C, int FORM>
__device__ __forceinline__ uint32_t SampleInsideCubicQ14(const Img &im, float sx, float sy)
{
    uint32_t r[4][C];
    LoadTapRows<C, 4, 4, FORM>(im, (int)floorf(sx), (int)floorf(sy), -1, -1, r);
    return BlendCubicQ14<C>(r, sx, sy);
}

// SampleWithBorder's fixed-point bilinear sum for a sample whose taps are all inside the image, whose
// coordinates are not negative and below 2^16, given in units of 2^-15 pixel: floor and fraction come
// from one float -> integer conversion, the taps of a row from one window, the two taps of a channel
// from one byte permute. Returns the pixel's dword.
template<int C, int FORM>
__device__ __forceinline__ uint32_t SampleInsideQ15(const Img &im, float sx, float sy)
{
    const uint32_t X = (uint32_t)(int)sx, Y = (uint32_t)(int)sy;
    const uint32_t ax = X & (kQ15 - 1), ay = Y & (kQ15 - 1);
    // WeightPairsQ15 with the sum 2^15 + 65535 ax as one instruction, its constant in a register (the compiler sees two
    // constants, which that instruction does not take, and writes one more; the resize kernels lose by it)
    const uint32_t bottom = __umul24((__umul24(ax, ay) + (kQ15 >> 1)) >> 15, 65535u) + ay;
    uint32_t       top;
    asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(top) : "v"(ax), "s"(65535u), "v"(kQ15));
    top -= bottom;
    uint32_t r[2][(2 * C + 3) / 4];
    LoadTapRows<C, 2, 2, FORM>(im, (int)(X >> 15), (int)(Y >> 15), 0, 0, r);
    uint32_t q = 0;
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        q = BlendQ15(BytePair(r[0], c, c + C), BytePair(r[1], c, c + C), top, bottom, c, q);
    }
    return q;
}

// SampleWithBorder's fixed-point bilinear sum for the two border modes that need no division - a constant
// colour (`constant`: borderPx, channel c in byte c) or the nearest pixel of the image -, straight-line: the
// four taps are fetched at coordinates clamped into the image and, for the constant border, replaced where the
// unclamped coordinate is outside. sx, sy in units of 2^-15 pixel, below 2^30 in magnitude. Same weights, same
// exact sum and the same single rounding as the generic path, so which path a sample takes does not show.
// The border modes' index maps for coordinates no farther than one image size outside the image (-(s - 1) .. 2s - 2
// for an axis of s pixels), where each is a single fold: index = c inside, k * c + lo in front, k * c + hi behind,
// with wave-uniform k, lo, hi per mode (DeviceUtils.hpp:BorderIndex for any coordinate, with its divisions):
//   constant, replicate  0 * c + 0      | 0 * c + s - 1     (the nearest pixel; the constant colour replaces it later)
//   reflect             -1 * c - 1      | -1 * c + 2s - 1
//   wrap                 1 * c + s      |  1 * c - s
//   reflect101          -1 * c          | -1 * c + 2s - 2
struct BorderFold
{
    int k, lo, hi, size;
};

__device__ __forceinline__ BorderFold MakeBorderFold(int border, int s)
{
    BorderFold f = {0, 0, s - 1, s};
    if (border == NVCV_BORDER_REFLECT)
    {
        f = {-1, -1, 2 * s - 1, s};
    }
    else if (border == NVCV_BORDER_WRAP)
    {
        f = {1, s, -s, s};
    }
    else if (border == NVCV_BORDER_REFLECT101)
    {
        f = {-1, 0, 2 * s - 2, s};
    }
    return f;
}

__device__ __forceinline__ int Fold(const BorderFold &f, int c)
{
    const int kc = f.k * c;
    return c < 0 ? kc + f.lo : (c >= f.size ? kc + f.hi : c);
}

// Pixel (x, y) of an 8-bit image, inside it, as a dword (channel c in byte c, the rest is not looked at): one
// 4-byte load, moved back where it would run past the image's last byte.
template<int C>
__device__ __forceinline__ uint32_t LoadPixelGuarded(const Img &im, uint32_t rowOffset, int x)
{
    const uint32_t lastLoad = (uint32_t)__mul24(im.h - 1, im.row) + (uint32_t)im.w * C - 4;
    const uint32_t at = rowOffset + (uint32_t)x * C, from = min(at, lastLoad);
    return LoadU32Unaligned(im.base + from) >> (8 * (at - from));
}

template<int C>
__device__ __forceinline__ uint32_t SampleNearBorderQ15(const Img &im, const BorderFold &fx, const BorderFold &fy, bool constant,
                                                        uint32_t borderPx, float sx, float sy)
{
    const int X = __float2int_rd(sx), Y = __float2int_rd(sy);
    const int x0 = X >> 15, y0 = Y >> 15;
    const int cx0 = Fold(fx, x0), cx1 = Fold(fx, x0 + 1);
    const uint32_t r0 = (uint32_t)__mul24(Fold(fy, y0), im.row), r1 = (uint32_t)__mul24(Fold(fy, y0 + 1), im.row);
    uint32_t p00 = LoadPixelGuarded<C>(im, r0, cx0), p01 = LoadPixelGuarded<C>(im, r0, cx1);
    uint32_t p10 = LoadPixelGuarded<C>(im, r1, cx0), p11 = LoadPixelGuarded<C>(im, r1, cx1);
    if (constant) // uniform
    {
        const bool inX0 = (uint32_t)x0 < (uint32_t)im.w, inX1 = (uint32_t)(x0 + 1) < (uint32_t)im.w;
        const bool inY0 = (uint32_t)y0 < (uint32_t)im.h, inY1 = (uint32_t)(y0 + 1) < (uint32_t)im.h;
        p00             = inX0 && inY0 ? p00 : borderPx;
        p01             = inX1 && inY0 ? p01 : borderPx;
        p10             = inX0 && inY1 ? p10 : borderPx;
        p11             = inX1 && inY1 ? p11 : borderPx;
    }
    return BilinearQ15<C>(p00, p01, p10, p11, (uint32_t)X & (kQ15 - 1), (uint32_t)Y & (kQ15 - 1));
}

// The same for the fixed-point bicubic sum: the 4 x 4 taps fetched at clamped coordinates (replaced by the colour
// where the unclamped one is outside), put together as the rows BlendCubicQ14 takes. |sx|, |sy| below 2^24.
template<int C>
__device__ __forceinline__ uint32_t SampleNearBorderCubicQ14(const Img &im, const BorderFold &fx, const BorderFold &fy,
                                                             bool constant, uint32_t borderPx, float sx, float sy)
{
    const int ix = (int)floorf(sx) - 1, iy = (int)floorf(sy) - 1;
    int       cx[4];
    bool      inX[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        cx[i]  = Fold(fx, ix + i);
        inX[i] = (uint32_t)(ix + i) < (uint32_t)im.w;
    }
    uint32_t r[4][C];
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        const uint32_t rowOffset = (uint32_t)__mul24(Fold(fy, iy + j), im.row);
        const bool     inY       = (uint32_t)(iy + j) < (uint32_t)im.h;
        uint32_t       p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            p[i] = LoadPixelGuarded<C>(im, rowOffset, cx[i]);
            if (constant) // uniform
            {
                p[i] = inX[i] && inY ? p[i] : borderPx;
            }
        }
        if constexpr (C == 3)
        {
            r[j][0] = __builtin_amdgcn_perm(p[1], p[0], 0x04020100u);
            r[j][1] = __builtin_amdgcn_perm(p[2], p[1], 0x05040201u);
            r[j][2] = __builtin_amdgcn_perm(p[3], p[2], 0x06050402u);
        }
        else if constexpr (C == 4)
        {
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                r[j][i] = p[i];
            }
        }
        else
        {
            r[j][0] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(p[3], p[2], 0x04000c0cu), __builtin_amdgcn_perm(p[1], p[0], 0x0c0c0400u),
                                            0x07060100u);
        }
    }
    return BlendCubicQ14<C>(r, sx, sy);
}

// Whether the image has room for the windows of SampleClampedCubicQ14. Where it has they pay at every size of launch, us with
// SampleNearBorderCubicQ14 / with windows, u8x3 under a replicating border: one 64 x 48 4.6 / 4.2, 200 x 150 4.7 / 4.7, 320 x 240 4.3 /
// 4.3 (in perspective 4.5 / 4.4), 400 x 300 5.7 / 5.1, 640 x 480 6.2 / 5.2, 1280 x 720 11.6 / 9.5; 40 x 16 x 16 4.4 / 4.0, 12 x 224 x 224 9.6 /
// 7.8; 32 x 1280 x 780 202 / 158.
template<int C>
__device__ __forceinline__ bool ClampedCubicFits(const Img &im)
{
    return im.w >= 4 && __mul24(im.h - 1, im.row) + im.w * C >= 16;
}

// SampleNearBorderCubicQ14 under a constant or replicating border: 4 loads per sample instead of 16. A row is the window of
// the 4 pixels nearest to the taps, and the taps' weights move instead of the pixels: each is added to the window pixel that
// its tap is clamped to or, under a constant border, taken out and given to the colour. The weights are integers, so the row
// sums stay the same integers. Replicating, perspective: 16 x 1240 x 1754 u8x3 164.2 -> 159.3 us, 24 x 1283 x 721 u8x1
// 86.3 -> 65.6 us, u8x4 58.4 -> 55.7 us.
template<int C>
__device__ __forceinline__ uint32_t SampleClampedCubicQ14(const Img &im, bool constant, uint32_t borderPx, float sx, float sy)
{
    typedef unsigned short U16x2 __attribute__((ext_vector_type(2)));
    const float fx = floorf(sx), fy = floorf(sy);
    const int   ix = (int)fx - 1, iy = (int)fy - 1;
    float       wx[4], wy[4];
    CubicCoeffsFused(sx - fx, 16384.f, wx);
    CubicCoeffsFused(sy - fy, 1.f / 16384.f, wy);
    uint32_t p01, p23;
    CubicWeightPairsQ14(wx, p01, p23);

    const int xs = min(max(ix, 0), im.w - 4);
    U16x2     w01 = {0, 0}, w23 = {0, 0}; // of the window's pixels
    int       kept = 0;                   // their sum
#pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        int w = (short)(i < 2 ? p01 >> (16 * i) : p23 >> (16 * (i - 2)));
        w     = constant && (uint32_t)(ix + i) >= (uint32_t)im.w ? 0 : w;
        kept += w;
        const int      at = min(max(i + (ix - xs), 0), 3);
        const uint64_t v  = (uint64_t)(uint32_t)(w & 0xffff) << (16 * at);
        const uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
        w01 += __builtin_bit_cast(U16x2, lo);
        w23 += __builtin_bit_cast(U16x2, hi);
    }
    p01 = __builtin_bit_cast(uint32_t, w01);
    p23 = __builtin_bit_cast(uint32_t, w23);

    constexpr bool kWindow = kWideTapLoads<uint8_t, C>;
    constexpr int  kLoad   = kWindow ? C + 1 : C;
    struct alignas(4) W
    {
        uint32_t d[kLoad];
    };
    const uint32_t mis = kWindow ? (uint32_t)reinterpret_cast<uintptr_t>(im.base) & 3u : 0u;
    // where the last window may start: its last dword is the one that holds the image's last byte
    const uint32_t lastAt = (((uint32_t)(__mul24(im.h - 1, im.row) + im.w * C - 1) + mis) & ~3u) - 4 * (kLoad - 1);
    const uint8_t *base   = im.base - mis;
    uint32_t       r[4][C];
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        const int      y = min(max(iy + j, 0), im.h - 1);
        const uint32_t o = (uint32_t)__mul24(y, im.row) + (uint32_t)(xs * C) + mis;
        if constexpr (kWindow)
        {
            // (a window that would pass the last dword holds its bytes from a dword on: it starts one earlier)
            const uint32_t at = min(o & ~3u, lastAt);
            const bool     moved = o - at >= 4;
            const W        w = *reinterpret_cast<const W *>(base + at);
#pragma unroll
            for (int i = 0; i < C; ++i)
            {
                const uint32_t v = __builtin_amdgcn_alignbyte(w.d[i + 1], w.d[i], o);
                r[j][i]          = moved ? w.d[i + 1] : v;
            }
        }
        else
        {
            const Vec<uint8_t, 4 * C> v = *reinterpret_cast<const Vec<uint8_t, 4 * C> *>(base + o);
            __builtin_memcpy(r[j], &v, 4 * C);
        }
    }

    int acc0[4], row01[4], row23[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        const bool none = constant && (uint32_t)(iy + j) >= (uint32_t)im.h; // the row is the colour
        row01[j]        = none ? 0 : (int)p01;
        row23[j]        = none ? 0 : (int)p23;
        acc0[j]         = constant ? (none ? 16384 : 16384 - kept) : 0; // the colour's share
    }
    uint32_t q = 0;
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        const int colour = (int)((borderPx >> (8 * c)) & 0xffu);
        float     acc = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            // (RowSumQ14's sum, on top of the colour's)
            int h = Dot2I16(BytePair(r[j], c, c + C), row01[j], __mul24(colour, acc0[j]) + 0x4B100000);
            h     = Dot2I16(BytePair(r[j], c + 2 * C, c + 3 * C), row23[j], h);
            const float hf = __int_as_float(h) - 9437184.f;
            acc            = j == 0 ? hf * wy[0] : __builtin_fmaf(hf, wy[j], acc);
        }
        q = __builtin_amdgcn_cvt_pk_u8_f32(acc, c, q);
    }
    return q;
}

// And for the nearest pixel.
template<int C>
__device__ __forceinline__ uint32_t SampleNearBorderNearest(const Img &im, const BorderFold &fx, const BorderFold &fy,
                                                            bool constant, uint32_t borderPx, float sx, float sy)
{
    const int      x = FloorToInt(sx + .5f), y = FloorToInt(sy + .5f);
    const uint32_t p = LoadPixelGuarded<C>(im, (uint32_t)__mul24(Fold(fy, y), im.row), Fold(fx, x));
    return constant && !((uint32_t)x < (uint32_t)im.w && (uint32_t)y < (uint32_t)im.h) ? borderPx : p;
}

// The dwords of the pixel that SampleInside gives; what lies above the pixel's bytes is not looked at. u8 channels are
// rounded, saturated and placed into their byte by one instruction each (v_cvt_pk_u8_f32 with a byte select and the dword
// so far), where packing converted bytes takes as many shifts and merges again. FORM: see LoadTapRows.
template<class T, int C, int INTERP, int FORM>
__device__ __forceinline__ void SampleInsidePacked(const Img &im, float sx, float sy, uint32_t (&w)[(C * sizeof(T) + 3) / 4])
{
    if constexpr (kFixedPoint<T, INTERP>)
    {
        w[0] = SampleInsideQ15<C, FORM>(im, sx, sy);
    }
    else if constexpr (kFixedPointCubic<T, INTERP>)
    {
        w[0] = SampleInsideCubicQ14<C, FORM>(im, sx, sy);
    }
    else if constexpr (std::is_same_v<T, uint8_t>)
    {
        uint32_t r[1][1];
        LoadTapRows<C, 1, 1, FORM>(im, (int)floorf(sx + .5f), (int)floorf(sy + .5f), 0, 0, r);
        w[0] = r[0][0];
    }
    else
    {
        T v[C];
        SampleInside<T, C, INTERP>(im, sx, sy, v);
#pragma unroll
        for (int d = 0; d < (int)((C * sizeof(T) + 3) / 4); ++d)
        {
            w[d] = 0;
        }
        __builtin_memcpy(w, v, C * sizeof(T));
    }
}

// True when every tap of the sample at (sx, sy) lies outside the image. For an integer k,
// floor(v) < k <=> v < k and floor(v) >= k <=> v >= k; NaN coordinates fail every comparison.
template<int INTERP>
__device__ __forceinline__ bool TapsOutside(const Img &im, float sx, float sy)
{
    if constexpr (INTERP == NVCV_INTERP_NEAREST)
    {
        // the tap is floor(v + .5)
        return (sx + .5f < 0.f) | (sx + .5f >= (float)im.w) | (sy + .5f < 0.f) | (sy + .5f >= (float)im.h);
    }
    constexpr float lo = INTERP == NVCV_INTERP_CUBIC ? 1.f : 0.f;
    constexpr float hi = INTERP == NVCV_INTERP_CUBIC ? 2.f : 1.f;
    return (sx < -hi) | (sx >= (float)im.w + lo) | (sy < -hi) | (sy >= (float)im.h + lo);
}

// SampleWithBorder for a sample whose taps all lie outside the image under NVCV_BORDER_CONSTANT: every tap is
// the border value, the weights and the order of the sum are the general sampler's, nothing is loaded.
template<class T, int C, int INTERP>
__device__ __forceinline__ void SampleAllOutside(const WarpArgs &a, float sx, float sy, T (&out)[C])
{
    float t[C], acc[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        t[c]   = (float)BorderValueAs<T>(a.bval[c]);
        acc[c] = 0.f;
    }
    if constexpr (INTERP == NVCV_INTERP_NEAREST || kFixedPoint<T, INTERP>)
    {
        // the tap itself; in fixed point the weights add up to exactly 1
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            out[c] = (T)t[c];
        }
        return;
    }
    else if constexpr (INTERP == NVCV_INTERP_LINEAR)
    {
        const int x1 = FloorToInt(sx), y1 = FloorToInt(sy);
        const int x2 = x1 + 1, y2 = y1 + 1;
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            const float wx = (i & 1) ? (sx - x1) : (x2 - sx);
            const float wy = (i >> 1) ? (sy - y1) : (y2 - sy);
            const float w  = wx * wy;
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                acc[c] += t[c] * w;
            }
        }
    }
    else if constexpr (kFixedPointCubic<T, INTERP>)
    {
        // every row sum is the border value times 2^14: the horizontal weights add up to exactly 1
        float wy[4];
        CubicCoeffsFused(sy - floorf(sy), 1.f / 16384.f, wy);
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            const float h = t[c] * 16384.f;
            float       v = h * wy[0];
            v             = __builtin_fmaf(h, wy[1], v);
            v             = __builtin_fmaf(h, wy[2], v);
            v             = __builtin_fmaf(h, wy[3], v);
            out[c]        = SaturateCast<T>(v);
        }
        return;
    }
    else
    {
        const int ix = FloorToInt(sx), iy = FloorToInt(sy);
        float     wx[4], wy[4];
        CubicWeights<T>(sx - ix, wx);
        CubicWeights<T>(sy - iy, wy);
#pragma unroll
        for (int cy = 0; cy < 4; ++cy)
        {
#pragma unroll
            for (int cx = 0; cx < 4; ++cx)
            {
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    acc[c] = AddTap<T, INTERP>(acc[c], t[c], wx[cx] * wy[cy]);
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        out[c] = SaturateCast<T>(acc[c]);
    }
}

// SampleWithBorder for a sample that NearBorderForm lets through: all taps are requested before the first is used, at indices
// folded into the image, and replaced by the colour where they were outside under a constant border. The weights and the order
// of the sum are SampleWithBorder's.
template<class T, int C, int INTERP>
__device__ __forceinline__ void SampleNearBorder(const Img &im, const WarpArgs &a, const BorderFold &fx, const BorderFold &fy, float sx,
                                                 float sy, T (&out)[C])
{
    constexpr int N = INTERP == NVCV_INTERP_CUBIC ? 4 : INTERP == NVCV_INTERP_LINEAR ? 2 : 1;
    const bool    constant = a.border == NVCV_BORDER_CONSTANT;
    const float   half = INTERP == NVCV_INTERP_NEAREST ? .5f : 0.f;
    const int     x1 = FloorToInt(sx + half), y1 = FloorToInt(sy + half), x = x1 - (N == 4), y = y1 - (N == 4);
    uint32_t      at[N];
    bool          inX[N];
#pragma unroll
    for (int i = 0; i < N; ++i)
    {
        at[i]  = (uint32_t)Fold(fx, x + i) * (uint32_t)sizeof(Vec<T, C>);
        inX[i] = (uint32_t)(x + i) < (uint32_t)im.w;
    }
    Vec<T, C> p[N][N];
#pragma unroll
    for (int j = 0; j < N; ++j)
    {
        const uint32_t row = (uint32_t)__mul24(Fold(fy, y + j), im.row);
#pragma unroll
        for (int i = 0; i < N; ++i)
        {
            p[j][i] = *reinterpret_cast<const Vec<T, C> *>(im.base + (row + at[i]));
        }
    }
    float t[N][N][C];
#pragma unroll
    for (int j = 0; j < N; ++j)
    {
        const bool inY = (uint32_t)(y + j) < (uint32_t)im.h;
#pragma unroll
        for (int i = 0; i < N; ++i)
        {
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                t[j][i][c] = constant && !(inX[i] && inY) ? (float)BorderValueAs<T>(a.bval[c]) : (float)p[j][i].v[c];
            }
        }
    }
    if constexpr (INTERP == NVCV_INTERP_NEAREST)
    {
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            out[c] = (T)t[0][0][c];
        }
    }
    else
    {
        float wx[4], wy[4], acc[C];
        if constexpr (INTERP == NVCV_INTERP_LINEAR)
        {
            wx[0] = (x1 + 1) - sx;
            wx[1] = sx - x1;
            wy[0] = (y1 + 1) - sy;
            wy[1] = sy - y1;
        }
        else
        {
            CubicWeights<T>(sx - x1, wx);
            CubicWeights<T>(sy - y1, wy);
        }
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            acc[c] = 0.f;
        }
#pragma unroll
        for (int j = 0; j < N; ++j)
        {
#pragma unroll
            for (int i = 0; i < N; ++i)
            {
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    acc[c] = AddTap<T, INTERP>(acc[c], t[j][i][c], wx[i] * wy[j]);
                }
            }
        }
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            out[c] = SaturateCast<T>(acc[c]);
        }
    }
}

// 8-bit pixels of 1, 3 or 4 channels have samplers of their own for samples next to the image's edge.
template<class T, int C>
constexpr bool kNearBorderForms = std::is_same_v<T, uint8_t> && (C == 1 || C == 3 || C == 4);

// Whether a lane's samples can take those or SampleNearBorder: an image within the 24-bit offsets (the caller's test; for the 8-bit
// forms also of 4 bytes or more), coordinates small enough for the samplers' integer conversions (8-bit bilinear: times 2^15
// below 2^30; else below 2^24) and, for the three modes that mirror or repeat the image, every tap no farther than one image
// size outside it (BorderFold; with a margin of two pixels for the widest tap window).
template<class T, int C, int INTERP, int N>
__device__ __forceinline__ bool NearBorderForm(const Img &im, const WarpArgs &a, const float (&sx)[N], const float (&sy)[N])
{
    constexpr float kScale = kCoordScale<T, INTERP>;
    uint32_t        u = 0;
    float           minX = sx[0], maxX = sx[0], minY = sy[0], maxY = sy[0];
#pragma unroll
    for (int k = 0; k < N; ++k)
    {
        u    = max(u, max(__float_as_uint(sx[k]) & 0x7fffffffu, __float_as_uint(sy[k]) & 0x7fffffffu));
        minX = fminf(minX, sx[k]);
        maxX = fmaxf(maxX, sx[k]);
        minY = fminf(minY, sy[k]);
        maxY = fmaxf(maxY, sy[k]);
    }
    bool ok = u < (kFixedPoint<T, INTERP> ? 0x4e800000u : 0x4b800000u)
           && (!kNearBorderForms<T, C> || __mul24(im.h - 1, im.row) + im.w * C >= 4);
    if (a.border > NVCV_BORDER_REPLICATE) // wave-uniform
    {
        // taps reach from floor(v) - 1 to floor(v) + 2 at most: all of them within -(s - 1) .. 2s - 2
        ok = ok && minX >= (float)(2 - im.w) * kScale && maxX < (float)(2 * im.w - 4) * kScale
          && minY >= (float)(2 - im.h) * kScale && maxY < (float)(2 * im.h - 4) * kScale;
    }
    return ok;
}

// The colour of a constant border as the dwords of a pixel.
template<class T, int C>
__device__ __forceinline__ void BorderDwords(const WarpArgs &a, uint32_t (&w)[(C * sizeof(T) + 3) / 4])
{
    T v[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        v[c] = BorderValueAs<T>(a.bval[c]);
    }
#pragma unroll
    for (int d = 0; d < (int)((C * sizeof(T) + 3) / 4); ++d)
    {
        w[d] = 0;
    }
    __builtin_memcpy(w, v, C * sizeof(T));
}

// Which launches' waves list their samples at the image's edge (WarpTile): none, those under a constant border, all. 8-bit
// bilinear and nearest samples are too few instructions for it (32 x 1280 x 780 u8x3 54 us, listed 60), and so is copying
// pixels. 8-bit bicubic ones pay where what lies all outside takes no part and with three channels (40 images of 443 .. 974 x 412 ..
// 446 64.3 -> 60.5, 16 x 201 x 332 in perspective 15.3 -> 12.5; one channel, 49 x 1139 x 681: 98 and, listed, 112; replicating, one
// 320 x 240 x 3 7.2 and 8.8, 25 x 283 x 733 x 4 31.3 and 32.6).
enum EdgeLists
{
    kNoLists,
    kConstantBorderLists,
    kAllLists
};

template<class T, int C, int INTERP>
constexpr EdgeLists kEdgeLists = INTERP == NVCV_INTERP_NEAREST        ? kNoLists
                               : !std::is_same_v<T, uint8_t>          ? kAllLists
                               : INTERP == NVCV_INTERP_CUBIC && C == 3 ? kConstantBorderLists
                                                                      : kNoLists;

// A listed sample that NearBorderForm lets through, as the dwords of its pixel.
template<class T, int C, int INTERP>
__device__ __forceinline__ void SampleNearEdge(const Img &im, const WarpArgs &a, uint32_t borderPx, float sx, float sy,
                                               uint32_t (&w)[(C * sizeof(T) + 3) / 4])
{
    const BorderFold foldX = MakeBorderFold(a.border, im.w), foldY = MakeBorderFold(a.border, im.h);
    if constexpr (!kNearBorderForms<T, C>)
    {
        T v[C];
        SampleNearBorder<T, C, INTERP>(im, a, foldX, foldY, sx, sy, v);
#pragma unroll
        for (int d = 0; d < (int)((C * sizeof(T) + 3) / 4); ++d)
        {
            w[d] = 0;
        }
        __builtin_memcpy(w, v, C * sizeof(T));
    }
    else
    {
        static_assert(INTERP == NVCV_INTERP_CUBIC && kEdgeLists<T, C, INTERP> == kConstantBorderLists);
        if (ClampedCubicFits<C>(im)) // uniform
        {
            w[0] = SampleClampedCubicQ14<C>(im, true, borderPx, sx, sy);
        }
        else
        {
            w[0] = SampleNearBorderCubicQ14<C>(im, foldX, foldY, true, borderPx, sx, sy);
        }
    }
}

// Whether single-channel taps are read alone, at any address, and not in windows of dwords: where lanes next to each other
// lie more along the source's columns than along its rows, and a window's second dword is another one to fetch for every
// lane. 16 x 1280 x 720 u8x1, windows / taps alone, at 0.3 rad 30.3 / 38.0 us bilinear, at 0.65 36.1 / 37.9, at 0.8 37.5 / 35.6, at a
// quarter turn 36.2 / 22.2 (4 x 1283 x 721, rows of odd pitch, 11.3 / 13.6, 13.2 / 12.9, 13.3 / 11.4, 11.5 / 8.5); bicubic, whose windows are
// two dwords for four taps, at 0.8 66.5 / 77.4, at 1.0 68.2 / 59.6, at a quarter turn 67.7 / 38.4. (Below the line the taps
// alone were measured with the row pitch added per lane.)
template<int INTERP>
__device__ __forceinline__ bool NarrowTapsPay(const float (&m)[9])
{
    return fabsf(m[3]) > (INTERP == NVCV_INTERP_LINEAR ? 1.f : 1.5f) * fabsf(m[0]);
}

// One block's tile of the destination image `dst` (tile coordinates tx, ty), all its threads.
template<class T, int C, int INTERP, bool PERSP, bool LIST, int N, int WAVES>
__device__ __forceinline__ void WarpTile(const Img &im, const WarpArgs &a, const float (&m)[9], uint8_t *dst, int dstRow,
                                         int dstW, int dstH, int tx, int ty)
{
    constexpr int PB = C * sizeof(T), D = (PB + 3) / 4;
    using B          = Block<N, WAVES>;

    // ---- gather: lane (lx, ly) of wave w samples its pixel in N patches (side by side: a
    // wave covers 8 N columns x 8 rows)
    const int wave = B::kWaves == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lx = threadIdx.x & (kPatch - 1),
              ly = (threadIdx.x >> 3) & (kPatch - 1);
    const int x0 = tx * B::kTileW + wave % B::kAcross * kWaveW<N>, y0 = ty * B::kTileH + wave / B::kAcross * kPatch;
    // m maps to source coordinates times kCoordScale; so do sx, sy and the limits
    constexpr float kScale = kCoordScale<T, INTERP>;
    const float     limX = InsideLimit<INTERP>(im.w, kTapOverrun<T, C, INTERP>) * kScale, limY = InsideLimit<INTERP>(im.h, 0) * kScale;
    int         px[N], py[N]; // the lane's destination pixels
    float       sx[N], sy[N];
    uint32_t    q[D][N]; // q[d][k]: dword d of this lane's pixel in patch k
    // rows too long or too many for 24-bit offset arithmetic go through the generic path
    // (and, in fixed point, coordinates too large for coordinate * 2^15 in 31 bits)
    const bool fits = (im.row | im.h) < (1 << 23) && (!kFixedPoint<T, INTERP> || (im.w | im.h) < (1 << 16));
#pragma unroll
    for (int k = 0; k < N; ++k)
    {
        // pixels of the tile beyond the image edge repeat the edge pixel's sample; they are never stored
        px[k] = min(x0 + k * kPatch + lx, dstW - 1);
        py[k] = min(y0 + ly, dstH - 1);
    }
    MapCoords<PERSP>(m, px, py, sx, sy);
    // the wave's pixels as rows, for the store (kPitch: neighbouring rows on other banks)
    constexpr int kPitch = kWaveW<N> * D + (D == 1 ? 8 : D == 2 ? 16 : D == 4 ? 24 : 0);
    __shared__ __align__(16) uint32_t room[B::kWaves][kPatch][kPitch];
    auto     &rows = room[wave];
    const int lane = threadIdx.x & 63;

    auto sampleInside = [&]()
    {
        uint32_t w[N][D];
        auto sample = [&](auto form)
        {
#pragma unroll
            for (int k = 0; k < N; ++k)
            {
                SampleInsidePacked<T, C, INTERP, decltype(form)::value>(im, sx[k], sy[k], w[k]);
            }
        };
        if (std::is_same_v<T, uint8_t> && C == 1 && INTERP != NVCV_INTERP_NEAREST && NarrowTapsPay<INTERP>(m)) // uniform
        {
            sample(std::integral_constant<int, kNarrowTaps>{});
        }
        else if (!kWideTapLoads<T, C> || INTERP == NVCV_INTERP_NEAREST || (im.row & 3) == 0) // uniform
        {
            sample(std::integral_constant<int, kSameRows>{});
        }
        else
        {
            sample(std::integral_constant<int, kOddRows>{});
        }
#pragma unroll
        for (int k = 0; k < N; ++k)
        {
#pragma unroll
            for (int d = 0; d < D; ++d)
            {
                q[d][k] = w[k][d];
            }
        }
    };
    auto place = [&](int k)
    {
#pragma unroll
        for (int d = 0; d < D; ++d)
        {
            rows[ly][(k * kPatch + lx) * D + d] = q[d][k];
        }
    };
    if constexpr (LIST)
    {
        static_assert(kEdgeLists<T, C, INTERP> != kNoLists && kScale == 1.f);
        // ---- a wave that the image's edge passes through: its samples at the edge, usually fewer than 64 of the 256, are listed and,
        // when all lanes have sampled as in the other waves (those with taps outside at a place inside), handed out to the
        // lanes again; what is all outside under a constant border takes the colour. Where every lane went through all its four
        // samples for one of them at the edge, such waves cost 2 to 5 times as much as others, and in a launch of small images a
        // third are such: 3 x 258 x 271 f32x1 bicubic 16.0 -> 6.7 us, 7 x 318 x 538 f32x4 bilinear 14.6 -> 9.6, 3 x 646 x 752 f32x1 bilinear
        // 9.7 -> 6.2, 40 x 1021 x 1523 of these 169 -> 145; 38 images of 75 .. 801 x 232 .. 359 u8x3 bicubic 36.3 -> 32.0.
        const bool whole  = __builtin_amdgcn_ballot_w64(!fits || !TapsInside<INTERP>(limX, limY, sx, sy)) == 0;
        __shared__ uint8_t list[B::kWaves][64 * N];
        uint32_t inside = 0xf, colour[D] = {}; // inside: bit k: sample k
        int      edges  = 0;
        if (!whole)
        {
            const bool constant = a.border == NVCV_BORDER_CONSTANT;
            BorderDwords<T, C>(a, colour);
            inside = 0;
#pragma unroll
            for (int k = 0; k < N; ++k)
            {
                const bool in  = fits && TapInside<INTERP>(limX, limY, sx[k], sy[k]);
                const bool out = constant && TapsOutside<INTERP>(im, sx[k], sy[k]);
                if (out)
                {
                    T        v[C];
                    uint32_t w[D] = {};
                    SampleAllOutside<T, C, INTERP>(a, sx[k], sy[k], v);
                    __builtin_memcpy(w, v, PB);
#pragma unroll
                    for (int d = 0; d < D; ++d)
                    {
                        rows[ly][(k * kPatch + lx) * D + d] = w[d];
                    }
                }
                const bool     edge = !in && !out && x0 + k * kPatch + lx < dstW && y0 + ly < dstH;
                const uint64_t mask = __builtin_amdgcn_ballot_w64(edge);
                if (edge)
                {
                    const int before = __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
                    list[wave][edges + before] = (uint8_t)(k * 64 + lane);
                }
                edges += __builtin_popcountll(mask);
                inside |= in ? 1u << k : 0u;
                sx[k] = in ? sx[k] : (INTERP == NVCV_INTERP_CUBIC ? 1.f : 0.f);
                sy[k] = in ? sy[k] : (INTERP == NVCV_INTERP_CUBIC ? 1.f : 0.f);
            }
            asm("" : "+v"(inside)); // (one register, not a mask for each sample)
        }

        if (__builtin_amdgcn_ballot_w64(inside != 0) != 0) // (then the place inside is one)
        {
            sampleInside();
        }
        if (whole)
        {
#pragma unroll
            for (int k = 0; k < N; ++k)
            {
                place(k);
            }
        }
        else
        {
#pragma unroll
            for (int k = 0; k < N; ++k)
            {
                if ((inside >> k) & 1)
                {
                    place(k);
                }
            }
            WaveExchangeFence();
            // The first `count` listed samples, 64 at a time (once for most waves that have any); `nearby`: those that NearBorderForm lets
            // through, the others move to the list's front. Returns how many these are.
            auto edgeSamples = [&](auto nearby, int count)
            {
                int others = 0;
#pragma nounroll
                for (int first = 0; first < count; first += 64)
                {
                    const bool listed = first + lane < count;
                    const int  id = list[wave][listed ? first + lane : first], at = (id >> 6) * kPatch + (id & (kPatch - 1)), line = (id >> 3) & (kPatch - 1);
                    float      bx[1], by[1];
                    MapCoord<PERSP>(m, x0 + at, y0 + line, bx[0], by[0]);
                    bool mine = listed;
                    if constexpr (nearby.value)
                    {
                        mine = listed && fits && NearBorderForm<T, C, INTERP>(im, a, bx, by);
                        if (const uint64_t mask = __builtin_amdgcn_ballot_w64(listed && !mine))
                        {
                            if (listed && !mine) // (to places that have been read)
                            {
                                const int before = __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
                                list[wave][others + before] = (uint8_t)id;
                            }
                            others += __builtin_popcountll(mask);
                        }
                    }
                    if (!mine)
                    {
                        continue;
                    }
                    uint32_t w[D] = {};
                    if constexpr (nearby.value)
                    {
                        SampleNearEdge<T, C, INTERP>(im, a, colour[0], bx[0], by[0], w);
                    }
                    else
                    {
                        T v[C];
                        SampleWithBorder<T, C, INTERP>(im, a, bx[0], by[0], v);
                        __builtin_memcpy(w, v, PB);
                    }
#pragma unroll
                    for (int d = 0; d < D; ++d)
                    {
                        rows[line][at * D + d] = w[d];
                    }
                }
                return others;
            };
            // (two loops: one with both samplers holds the registers of both)
            const int others = edgeSamples(std::true_type{}, edges);
            WaveExchangeFence();
            edgeSamples(std::false_type{}, others);
        }
    }
    else
    {
        // Each lane takes its own samples, all in flight.
        bool in = fits & TapsInside<INTERP>(limX, limY, sx, sy);
        if constexpr (kFixedPointCubic<T, INTERP>)
        {
            // Where the windows that move their weights are taken, they serve the samples inside as well (the same integers): a wave
            // that the edge passes through goes through them alone, no longer through both forms. Kernel us before / after, replicating:
            // u8x4 32 x 256 x 256 18.7 / 15.5, 4 x 640 x 480 11.0 / 9.8, 16 x 1240 x 1754 in perspective 184 / 173; u8x3 32 x 256 x 256 21.3 / 19.3, 4 x 640 x
            // 480 12.0 / 11.2; u8x1 12.7 / 11.7, 7.4 / 7.0. (Listing the samples at the edge, as float images do: u8x3 26.6 and 14.0.)
            if (a.border <= NVCV_BORDER_REPLICATE && ClampedCubicFits<C>(im)) // uniform
            {
                in = __builtin_amdgcn_ballot_w64(!in) == 0;
            }
        }
        if constexpr (kFixedPoint<T, INTERP> && C != 1)
        {
            // The same for bilinear samples, whose form at the edge gives the same sum. us a call: 64 x 256 x 256 u8x3 constant border
            // 15.7 / 13.9, replicating 17.3 / 16.0, u8x4 16.5 / 15.4; 8 x 640 x 480 u8x3 9.2 / 7.7; 40 rotated images of 240 .. 480 16.0 / 15.3. One
            // channel, whose four single taps take twice the loads of its two windows, loses: 13.5 / 13.9, replicating 16.0 / 16.3.
            in = __builtin_amdgcn_ballot_w64(!in) == 0;
        }
        if (in)
        {
            sampleInside();
        }
        else if ((kNearBorderForms<T, C> || INTERP == NVCV_INTERP_NEAREST) && fits && NearBorderForm<T, C, INTERP>(im, a, sx, sy))
        {
            uint32_t colour[D];
            BorderDwords<T, C>(a, colour);
            // under a constant border a lane whose samples lie outside with all their taps needs no pixel: whole
            // waves in the corners a rotation leaves empty
            const bool       constant = a.border == NVCV_BORDER_CONSTANT;
            const BorderFold foldX = MakeBorderFold(a.border, im.w), foldY = MakeBorderFold(a.border, im.h);
            bool             outside = constant;
#pragma unroll
            for (int k = 0; k < N; ++k)
            {
                outside &= TapsOutside<INTERP>(im, sx[k] * (1.f / kScale), sy[k] * (1.f / kScale));
            }
            if (outside)
            {
#pragma unroll
                for (int k = 0; k < N; ++k)
                {
                    if constexpr (kFixedPointCubic<T, INTERP>)
                    {
                        T v[C];
                        SampleAllOutside<T, C, INTERP>(a, sx[k], sy[k], v);
                        q[0][k] = 0;
                        __builtin_memcpy(&q[0][k], v, C);
                        // (a dword from here on: the compiler carried its bytes apart through all paths, 28 instructions)
                        asm("" : "+v"(q[0][k]));
                    }
                    else
                    {
#pragma unroll
                        for (int d = 0; d < D; ++d)
                        {
                            q[d][k] = colour[d]; // the tap itself, or taps whose weights add up to exactly 1
                        }
                    }
                }
            }
            else if (INTERP == NVCV_INTERP_CUBIC && a.border <= NVCV_BORDER_REPLICATE && ClampedCubicFits<C>(im)) // uniform
            {
                // one sample at a time (all four at once took 143 registers, which every wave of the launch would have held;
                // held to the 64 of full occupancy the u8x3 kernel spills and loses 1 to 2 %)
#pragma nounroll
                for (int k = 0; k < N; ++k)
                {
                    float bx = sx[0], by = sy[0];
#pragma unroll
                    for (int j = 1; j < N; ++j)
                    {
                        bx = k == j ? sx[j] : bx;
                        by = k == j ? sy[j] : by;
                    }
                    // (a copy for each border: in one, the replicating border does the colour's share of the work as well; 32 x 256 x
                    // 256 u8x1 11.9 us in one copy, 10.0 in two, 4 x 1283 x 721 u8x3 27.4 and 25.9)
                    uint32_t v;
                    if (constant)
                    {
                        v = SampleClampedCubicQ14<C>(im, true, colour[0], bx, by);
                    }
                    else
                    {
                        v = SampleClampedCubicQ14<C>(im, false, colour[0], bx, by);
                    }
#pragma unroll
                    for (int j = 0; j < N; ++j)
                    {
                        q[0][j] = k == j ? v : q[0][j];
                    }
                }
            }
            else
            {
#pragma unroll
                for (int k = 0; k < N; ++k)
                {
                    if constexpr (kFixedPoint<T, INTERP>)
                    {
                        q[0][k] = SampleNearBorderQ15<C>(im, foldX, foldY, constant, colour[0], sx[k], sy[k]);
                    }
                    else if constexpr (kFixedPointCubic<T, INTERP>)
                    {
                        q[0][k] = SampleNearBorderCubicQ14<C>(im, foldX, foldY, constant, colour[0], sx[k], sy[k]);
                    }
                    else if constexpr (kNearBorderForms<T, C>)
                    {
                        q[0][k] = SampleNearBorderNearest<C>(im, foldX, foldY, constant, colour[0], sx[k], sy[k]);
                    }
                    else
                    {
                        T        v[C];
                        uint32_t w[D] = {};
                        SampleNearBorder<T, C, INTERP>(im, a, foldX, foldY, sx[k], sy[k], v);
                        __builtin_memcpy(w, v, PB);
#pragma unroll
                        for (int d = 0; d < D; ++d)
                        {
                            q[d][k] = w[d];
                        }
                    }
                }
            }
        }
        else
        {
#pragma nounroll
            for (int k = 0; k < N; ++k)
            {
                // position and coordinates recomputed rather than indexed, results placed by selects: a
                // run-time index would put the arrays in scratch memory
                const int dx = min(x0 + k * kPatch + lx, dstW - 1), dy = min(y0 + ly, dstH - 1);
                float     bx, by;
                MapCoord<PERSP>(m, dx, dy, bx, by);
                bx *= 1.f / kScale;
                by *= 1.f / kScale;
                T v[C];
                if (a.border == NVCV_BORDER_CONSTANT && TapsOutside<INTERP>(im, bx, by))
                {
                    SampleAllOutside<T, C, INTERP>(a, bx, by, v);
                }
                else
                {
                    SampleWithBorder<T, C, INTERP>(im, a, bx, by, v);
                }
                uint32_t w[D] = {};
                __builtin_memcpy(w, v, PB);
#pragma unroll
                for (int d = 0; d < D; ++d)
                {
                    asm("" : "+v"(w[d]));
#pragma unroll
                    for (int j = 0; j < N; ++j)
                    {
                        q[d][j] = k == j ? w[d] : q[d][j];
                    }
                }
            }
        }
#pragma unroll
        for (int k = 0; k < N; ++k)
        {
            place(k);
        }
    }
    WaveExchangeFence();

    // ---- store. Pixels of 12 and 16 bytes leave as the rows they form, 16 bytes per lane: 384 or 512 contiguous bytes of each
    // row. One pixel per lane wrote 96 or 128 bytes of 8 rows per instruction, with a partly written sector at both ends of
    // most: 4 x 1283 x 721 f32x3 nearest 30.5 -> 19.4 us, bilinear 28.4 -> 24.3; f32x4 33.1 -> 22.0 and 30.4 -> 27.3 (of rows that
    // start at sectors, 1280 x 720: f32x3 22.3 -> 16.6, f32x4 5 % slower when small, one 1280 x 720 5.4 -> 5.7, and as before when
    // large; a second form of the store for these cost all others 3 to 5 %).
    if constexpr (PB >= 12)
    {
        constexpr int kChunks = kWaveW<N> * PB / 16;
        const int dwords = min(dstW - x0, kWaveW<N>) * D; // of a row
        uint8_t  *to = dst + (int64_t)y0 * dstRow + (int64_t)x0 * PB;
#pragma unroll
        for (int i = 0; i < (kPatch * kChunks + 63) / 64; ++i)
        {
            const int row = (lane + 64 * i) / kChunks, at = (lane + 64 * i) % kChunks * 4;
            if (y0 + row >= dstH || at >= dwords || (kPatch * kChunks % 64 != 0 && row >= kPatch))
            {
                continue;
            }
            const uint4    v    = *reinterpret_cast<const uint4 *>(&rows[row][at]);
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
            uint8_t       *p    = to + (uint32_t)(row * dstRow + at * 4);
            if (at + 4 <= dwords)
            {
                StoreDwordsNT<4>(p, w);
            }
            else
            {
#pragma unroll
                for (int d = 0; d < 3; ++d)
                {
                    if (at + d < dwords)
                    {
                        const uint32_t one[1] = {w[d]};
                        StoreDwordsNT<1>(p + 4 * d, one);
                    }
                }
            }
        }
        return;
    }
    // Of smaller pixels lane (lx, ly) stores columns 4 lx .. 4 lx + 3 of row ly. (Through LDS: these kernels wait for vector
    // instructions; moves and selects between lanes took 20 for each dword of a pixel, and left a row's pieces in another
    // order than the lanes'.)
    const int dx0 = x0 + 4 * lx;
    uint32_t  quad[D][4] = {};
    if (N < kMostPatches && lx >= kWaveW<N> / 4)
    {
        return;
    }
    if constexpr (PB < 12)
    {
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
#pragma unroll
            for (int d = 0; d < D; ++d)
            {
                quad[d][k] = rows[ly][(4 * lx + k) * D + d];
            }
        }
    }
    const int dy = y0 + ly;
    if (dy >= dstH || dx0 >= dstW)
    {
        return;
    }
    // (the wave's rows start at one address, and a lane's bytes are less than 2 GiB behind it: an image's are)
    uint8_t *to = dst + (int64_t)y0 * dstRow + (int64_t)x0 * PB + (uint32_t)(ly * dstRow + (dx0 - x0) * PB);
    if (dx0 + 4 <= dstW)
    {
        uint32_t w[PB];
        PackQuad<PB>(quad, w);
        // (one channel too, whose 32 bytes of a row are mostly parts of sectors: by ordinary stores, which the L2 puts together, 400 launches take 0.97 of
        // the time for nearest neighbour and 1.00 for bilinear while inputs and outputs stay in the memory's cache, but 1.04 and 1.03, up to 1.28, where they do not)
        StoreDwordsNT<PB>(to, w); // 4 pixels = PB dwords
    }
    else
    {
#pragma unroll
        for (int k = 0; k < 3; ++k)
        {
            if (dx0 + k < dstW)
            {
                uint32_t w[D];
#pragma unroll
                for (int d = 0; d < D; ++d)
                {
                    w[d] = quad[d][k];
                }
                Vec<T, C> px;
                __builtin_memcpy(&px, w, PB);
                reinterpret_cast<Vec<T, C> *>(to)[k] = px;
            }
        }
    }
}

// Loads image `image`'s matrix from the caller's tensor and, unless it already maps destination to
// source, inverts it (uniform per block). The first two rows come out multiplied by `scale` (a power of
// two: scaling commutes with every rounding of the products and sums that form a coordinate, so
// coordinates computed from the scaled rows are the scaled coordinates bit for bit).
template<bool PERSP>
__device__ __forceinline__ void LoadMatrix(const WarpArgs &a, int image, float scale, float (&m)[9])
{
    const float *p = reinterpret_cast<const float *>(a.xforms + image * a.xformStride);
    float        f[9];
#pragma unroll
    for (int i = 0; i < 9; ++i)
    {
        f[i] = i < (PERSP ? 9 : 6) ? p[i] : 0.f;
    }
    if (a.inverseGiven != 0)
    {
        m[0] = f[0] * scale;
        m[1] = f[1] * scale;
        m[2] = f[2] * scale;
        m[3] = f[3] * scale;
        m[4] = f[4] * scale;
        m[5] = f[5] * scale;
        m[6] = f[6];
        m[7] = f[7];
        m[8] = f[8];
    }
    else if constexpr (!PERSP)
    {
        // affine inverse (reference: warp.cu:139-150, 1/det evaluated in double and rounded to float32, which
        // is what the correctly rounded float32 quotient gives; 1e-5 there is a double: for a float32
        // operand, greater than it means greater than the float32 just below it)
        float den = f[0] * f[4] - f[1] * f[3];
        den       = (fabsf(den) > 9.99999974738e-06f ? 1.f / den : 0.f) * scale;
        m[0]      = f[4] * den;
        m[1]      = -f[1] * den;
        m[2]      = (f[1] * f[5] - f[4] * f[2]) * den;
        m[3]      = -f[3] * den;
        m[4]      = f[0] * den;
        m[5]      = (f[3] * f[2] - f[0] * f[5]) * den;
        m[6] = m[7] = m[8] = 0.f;
    }
    else
    {
        // 3x3 inverse by cofactors (reference: cuda_tools/math/LinAlg.hpp:1446-1450, 1640-1654); a singular
        // matrix is left as given, like the reference's failed in-place inverse
        const float d = f[0] * (f[4] * f[8] - f[5] * f[7]) + f[1] * (f[5] * f[6] - f[3] * f[8])
                      + f[2] * (f[3] * f[7] - f[4] * f[6]);
        const bool  ok = d != 0;
        m[0]           = (ok ? (f[4] * f[8] - f[5] * f[7]) / d : f[0]) * scale;
        m[1]           = (ok ? -(f[1] * f[8] - f[2] * f[7]) / d : f[1]) * scale;
        m[2]           = (ok ? (f[1] * f[5] - f[2] * f[4]) / d : f[2]) * scale;
        m[3]           = (ok ? -(f[3] * f[8] - f[5] * f[6]) / d : f[3]) * scale;
        m[4]           = (ok ? (f[0] * f[8] - f[2] * f[6]) / d : f[4]) * scale;
        m[5]           = (ok ? -(f[0] * f[5] - f[2] * f[3]) / d : f[5]) * scale;
        m[6]           = ok ? (f[3] * f[7] - f[4] * f[6]) / d : f[6];
        m[7]           = ok ? -(f[0] * f[7] - f[1] * f[6]) / d : f[7];
        m[8]           = ok ? (f[0] * f[4] - f[1] * f[3]) / d : f[8];
    }
}

template<class T, int C, int INTERP, bool PERSP, bool LIST, int PATCHES, int WAVES>
__global__ __launch_bounds__((64 * WAVES)) void WarpTensor(const WarpArgs a)
{
    const int n  = blockIdx.z;
    const Img im = {a.src + n * a.srcN, a.srcRow, a.srcW, a.srcH};
    float     m[9];
#pragma unroll
    for (int i = 0; i < 9; ++i)
    {
        m[i] = a.m[i];
    }
    WarpTile<T, C, INTERP, PERSP, LIST, PATCHES, WAVES>(im, a, m, a.dst + n * a.dstN, a.dstRow, a.dstW, a.dstH, blockIdx.x, blockIdx.y);
}

template<class T, int C, int INTERP, bool PERSP, bool LIST, int PATCHES, int WAVES>
__global__ __launch_bounds__((64 * WAVES)) void WarpVarShape(const WarpArgs a, const VarTiles tiles)
{
    const TileCoord tc = LocateTile(tiles, blockIdx.x);
    // descriptors and matrix depend on the image index only: read by value here, ahead of the matrix
    // arithmetic, so that all of these loads share one memory round trip
    const NVCVImagePlaneStrided s = a.srcList[tc.image].planes[0];
    const NVCVImagePlaneStrided d = a.dstList[tc.image].planes[0];
    float                       m[9];
    LoadMatrix<PERSP>(a, tc.image, kCoordScale<T, INTERP>, m);
    const Img im = {AsGlobal(s.basePtr), s.rowStride, s.width, s.height};
    WarpTile<T, C, INTERP, PERSP, LIST, PATCHES, WAVES>(im, a, m, AsGlobal(d.basePtr), d.rowStride, d.width, d.height, tc.tx, tc.ty);
}

// Two patches per wave instead of four where that leaves a SIMD no more than 3 waves of four: such launches run as long as one
// wave does, whose four samples a lane follow one another in issue, and half of it is done in little more than half the
// time. From about 5 waves per SIMD on the waves' own start (matrix, tile search, edge tests) is what counts. Kernel us with four / two
// patches, under a constant border: u8x3 bicubic 320 x 240 8.8 / 6.0, 640 x 480 8.8 / 6.6, 2 of them (2 400 waves) 8.0 / 7.0, 4 10.6 / 10.0,
// 8 15.1 / 15.5, 16 24.9 / 27.0; bilinear 4.6 / 3.8, 5.1 / 4.1, 5.3 / 4.6, 6.1 / 6.0, 8.8 / 8.7, 13.4 / 14.4; f32x4 bicubic 7.6 / 5.4, 8.0 / 7.0, 10.0 /
// 9.3, 14.6 / 13.4; f32x1 bilinear 4.4 / 3.8, 4.6 / 4.4, 4.6 / 4.4, 5.3 / 5.5, 7.2 / 7.8; u8x3 nearest 3.8 / 3.4, 3.8 / 3.3, 4.2 / 3.9, 4.6 / 4.8.
// (One patch: 320 x 240 u8x3 bicubic 5.2, but 2 x 640 x 480 7.4 and 16 30.5; elements of 16 bits keep four, for the size of the library.)
constexpr int64_t kFewWaves = 3 * 1024;
// Waves of image batches start with the tile search and the matrix' inversion as well, so the line lies lower where the samples are
// few instructions. Two patches over four by numbers of waves, means over 700 random launches: nearest neighbour up to 1 536 0.95,
// to 2 048 0.99, to 2 560 1.01 (in perspective 1.04), to 3 072 1.02 (60 of 48 x 176 u8x4 in perspective 6.1 us with four and 7.05 with
// two); 8-bit bilinear in perspective to 2 560 0.92, to 3 072 1.02; bilinear of floats to 3 072 0.93, bicubic 0.90.
template<class T, int INTERP, bool PERSP>
constexpr int64_t kFewWavesOfBatches = INTERP == NVCV_INTERP_NEAREST                                    ? 1536
                                     : INTERP == NVCV_INTERP_LINEAR && PERSP && std::is_same_v<T, uint8_t> ? 2560
                                                                                                        : kFewWaves;
template<class T>
constexpr bool kFewPatchesForm = std::is_same_v<T, uint8_t> || std::is_same_v<T, float>;

template<class T, int C, int INTERP, bool PERSP, bool LIST>
void LaunchMap(const WarpArgs &a, int N, const NVCVImageBufferStrided *dstHost, hipStream_t stream)
{
    constexpr int kMost = kMostPatches, kFew = kFewPatchesForm<T> ? kFewPatches : kMost;
    using Four          = Block<kMost, 4>;
    using Few           = Block<kFew, 4>;
    using One           = Block<kMost, kSingleWaves<T, C, INTERP, kMost> ? 1 : 4>;
    const auto few  = [](int64_t tiles, int64_t most) { return kFew != kMost && tiles * Four::kWaves <= most; };
    const auto ones = [](int64_t one, int64_t four) { return One::kWaves == 1 && SingleWavesPay(one, four * Four::kWaves); };
    if (dstHost == nullptr)
    {
        const auto    gridOf = [&](int w, int h) { return dim3(DivUp(a.dstW, w), DivUp(a.dstH, h), N); };
        const auto    count  = [&](int w, int h) { return (int64_t)DivUp(a.dstW, w) * DivUp(a.dstH, h) * N; };
        const int64_t four   = count(Four::kTileW, Four::kTileH);
        if (few(four, kFewWaves))
        {
            hipLaunchKernelGGL((WarpTensor<T, C, INTERP, PERSP, LIST, kFew, 4>), gridOf(Few::kTileW, Few::kTileH), dim3(Few::kThreads), 0, stream, a);
        }
        else if (ones(count(One::kTileW, One::kTileH), four))
        {
            hipLaunchKernelGGL((WarpTensor<T, C, INTERP, PERSP, LIST, kMost, One::kWaves>), gridOf(One::kTileW, One::kTileH), dim3(One::kThreads), 0,
                               stream, a);
        }
        else
        {
            hipLaunchKernelGGL((WarpTensor<T, C, INTERP, PERSP, LIST, kMost, 4>), gridOf(Four::kTileW, Four::kTileH), dim3(Four::kThreads), 0, stream, a);
        }
        CheckLaunch("WarpTensor");
        return;
    }
    for (int first = 0; first < N; first += kMaxTileImages)
    {
        VarTiles   tiles;
        const int  count   = std::min(kMaxTileImages, N - first);
        const auto totalOf = [&](int w, int h) { return BuildVarTiles(tiles, dstHost, first, count, w, h); };
        const auto tilesOf = [&](int w, int h)
        {
            int64_t sum = 0;
            for (int i = first; i < first + count; ++i)
            {
                sum += (int64_t)DivUp(dstHost[i].planes[0].width, w) * DivUp(dstHost[i].planes[0].height, h);
            }
            return sum;
        };
        const int64_t four = tilesOf(Four::kTileW, Four::kTileH);
        if (four <= 0)
        {
            continue;
        }
        if (few(four, kFewWavesOfBatches<T, INTERP, PERSP>))
        {
            const int total = totalOf(Few::kTileW, Few::kTileH);
            hipLaunchKernelGGL((WarpVarShape<T, C, INTERP, PERSP, LIST, kFew, 4>), dim3(total), dim3(Few::kThreads), 0, stream, a, tiles);
        }
        else if (One::kWaves == 1 && ones(tilesOf(One::kTileW, One::kTileH), four))
        {
            const int total = totalOf(One::kTileW, One::kTileH);
            hipLaunchKernelGGL((WarpVarShape<T, C, INTERP, PERSP, LIST, kMost, One::kWaves>), dim3(total), dim3(One::kThreads), 0, stream, a, tiles);
        }
        else
        {
            const int total = totalOf(Four::kTileW, Four::kTileH);
            hipLaunchKernelGGL((WarpVarShape<T, C, INTERP, PERSP, LIST, kMost, 4>), dim3(total), dim3(Four::kThreads), 0, stream, a, tiles);
        }
        CheckLaunch("WarpVarShape");
    }
}

template<class T, int C, int INTERP>
void Launch(const WarpArgs &a, int N, const NVCVImageBufferStrided *dstHost, hipStream_t stream)
{
    constexpr EdgeLists kLists = kEdgeLists<T, C, INTERP>;
    if (kLists == kAllLists || (kLists == kConstantBorderLists && a.border == NVCV_BORDER_CONSTANT))
    {
        constexpr bool kList = kLists != kNoLists;
        a.perspective ? LaunchMap<T, C, INTERP, true, kList>(a, N, dstHost, stream) : LaunchMap<T, C, INTERP, false, kList>(a, N, dstHost, stream);
    }
    else
    {
        constexpr bool kList = kLists == kAllLists;
        a.perspective ? LaunchMap<T, C, INTERP, true, kList>(a, N, dstHost, stream) : LaunchMap<T, C, INTERP, false, kList>(a, N, dstHost, stream);
    }
}

template<class T, int C>
void DispatchInterp(int interp, const WarpArgs &a, int N, const NVCVImageBufferStrided *dstHost, hipStream_t stream)
{
    switch (interp)
    {
    case NVCV_INTERP_NEAREST:
        Launch<T, C, NVCV_INTERP_NEAREST>(a, N, dstHost, stream);
        break;
    case NVCV_INTERP_LINEAR:
        Launch<T, C, NVCV_INTERP_LINEAR>(a, N, dstHost, stream);
        break;
    case NVCV_INTERP_CUBIC:
        Launch<T, C, NVCV_INTERP_CUBIC>(a, N, dstHost, stream);
        break;
    default:
        throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Invalid interpolation (supported: NEAREST, LINEAR, CUBIC)");
    }
}

template<class T>
void DispatchC(int C, int interp, const WarpArgs &a, int N, const NVCVImageBufferStrided *dstHost, hipStream_t stream)
{
    switch (C)
    {
    case 1:
        DispatchInterp<T, 1>(interp, a, N, dstHost, stream);
        break;
    case 3:
        DispatchInterp<T, 3>(interp, a, N, dstHost, stream);
        break;
    case 4:
        DispatchInterp<T, 4>(interp, a, N, dstHost, stream);
        break;
    default:
        throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Invalid channel number %d", C);
    }
}

void DispatchType(ElemType e, int C, int interp, const WarpArgs &a, int N, const NVCVImageBufferStrided *dstHost,
                  hipStream_t stream)
{
    if (N == 0)
    {
        return;
    }
    switch (e)
    {
    case kU8:
        DispatchC<uint8_t>(C, interp, a, N, dstHost, stream);
        break;
    case kU16:
        DispatchC<uint16_t>(C, interp, a, N, dstHost, stream);
        break;
    case kS16:
        DispatchC<int16_t>(C, interp, a, N, dstHost, stream);
        break;
    case kF32:
        DispatchC<float>(C, interp, a, N, dstHost, stream);
        break;
    default:
        throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Invalid DataType");
    }
}

void CheckBorder(NVCVBorderType b)
{
    if ((int)b < NVCV_BORDER_CONSTANT || (int)b > NVCV_BORDER_REFLECT101)
    {
        throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Invalid border mode %d", (int)b);
    }
}

void InvertAffineHost(const float *M, float *out)
{
    float den = M[0] * M[4] - M[1] * M[3];
    den       = std::abs(den) > 1e-5 ? 1. / den : .0;
    out[0]    = (float)M[4] * den;
    out[1]    = (float)-M[1] * den;
    out[2]    = (float)(M[1] * M[5] - M[4] * M[2]) * den;
    out[3]    = (float)-M[3] * den;
    out[4]    = (float)M[0] * den;
    out[5]    = (float)(M[3] * M[2] - M[0] * M[5]) * den;
    out[6] = out[7] = out[8] = 0.f;
}

void InvertPerspectiveHost(const float *f, float *m)
{
    const float d
        = f[0] * (f[4] * f[8] - f[5] * f[7]) + f[1] * (f[5] * f[6] - f[3] * f[8]) + f[2] * (f[3] * f[7] - f[4] * f[6]);
    if (d == 0)
    {
        std::copy_n(f, 9, m);
        return;
    }
    m[0] = (f[4] * f[8] - f[5] * f[7]) / d;
    m[1] = -(f[1] * f[8] - f[2] * f[7]) / d;
    m[2] = (f[1] * f[5] - f[2] * f[4]) / d;
    m[3] = -(f[3] * f[8] - f[5] * f[6]) / d;
    m[4] = (f[0] * f[8] - f[2] * f[6]) / d;
    m[5] = -(f[0] * f[5] - f[2] * f[3]) / d;
    m[6] = (f[3] * f[7] - f[4] * f[6]) / d;
    m[7] = -(f[0] * f[7] - f[1] * f[6]) / d;
    m[8] = (f[0] * f[4] - f[1] * f[3]) / d;
}

class Warp : public IOperator
{
public:
    Warp(bool perspective, int32_t maxVarShapeBatchSize)
        : m_perspective(perspective)
        , m_maxBatch(maxVarShapeBatchSize)
    {
        if (maxVarShapeBatchSize < 0)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "maxVarShapeBatchSize must be >= 0");
        }
    }

    void submit(hipStream_t stream, NVCVTensorHandle hin, NVCVTensorHandle hout, const float *xform, int32_t flags,
                NVCVBorderType border, float4 bval) const
    {
        if (xform == nullptr)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Transformation matrix must not be NULL");
        }
        NVCVTensorData din, dout;
        ExportTensor(hin, din, "Input");
        ExportTensor(hout, dout, "Output");
        ImageBatchView in  = RequireImageBatchView(din, "Input", NVCV_ERROR_INVALID_ARGUMENT);
        ImageBatchView out = RequireImageBatchView(dout, "Output", NVCV_ERROR_INVALID_ARGUMENT);
        if (in.layout != kLayoutNHWC || out.layout != kLayoutNHWC || in.hasBatchDim != out.hasBatchDim)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT,
                          "Invalid DataFormat between input (%s) and output (%s): both must be \"NHWC\" or \"HWC\"",
                          in.layoutName, out.layoutName);
        }
        if (in.C > 4)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Invalid channel number %d", in.C);
        }
        if (in.elem != out.elem || in.C != out.C || in.N != out.N)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT,
                          "Input and output must have the same data type, channel count and batch size");
        }
        if (std::max(in.bytesSpanned(), out.bytesSpanned()) > INT32_MAX)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Input or output size exceeds %d. Tensor is too large.",
                          INT32_MAX);
        }
        CheckBorder(border);
        WarpArgs a = makeArgs(border, bval);
        if (flags & NVCV_WARP_INVERSE_MAP)
        {
            for (int i = 0; i < 9; ++i)
            {
                a.m[i] = i < (m_perspective ? 9 : 6) ? xform[i] : 0.f;
            }
        }
        else if (m_perspective)
        {
            InvertPerspectiveHost(xform, a.m);
        }
        else
        {
            InvertAffineHost(xform, a.m);
        }
        if (in.elem == kU8 && (flags & NVCV_INTERP_MAX) == NVCV_INTERP_LINEAR)
        {
            for (int i = 0; i < 6; ++i)
            {
                a.m[i] *= kCoordScale<uint8_t, NVCV_INTERP_LINEAR>; // see kCoordScale
            }
        }
        a.src    = in.base;
        a.dst    = out.base;
        a.srcN   = in.strideN;
        a.dstN   = out.strideN;
        a.srcRow = (int32_t)in.strideH;
        a.dstRow = (int32_t)out.strideH;
        a.srcW   = in.W;
        a.srcH   = in.H;
        a.dstW   = out.W;
        a.dstH   = out.H;
        if (out.W == 0 || out.H == 0 || in.W == 0 || in.H == 0)
        {
            return;
        }
        DispatchType(in.elem, in.C, flags & NVCV_INTERP_MAX, a, in.N, nullptr, stream);
    }

    void submit(hipStream_t stream, NVCVImageBatchHandle hin, NVCVImageBatchHandle hout, NVCVTensorHandle hxform,
                int32_t flags, NVCVBorderType border, float4 bval) const
    {
        if (m_maxBatch <= 0)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT,
                          "Operator was not created for var-shape use, maxVarShapeBatchSize: %d", m_maxBatch);
        }
        VarShapeView in  = ExportVarShape(hin, stream, "Input");
        VarShapeView out = ExportVarShape(hout, stream, "Output");
        if (in.N > m_maxBatch)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Invalid number of images, it should not exceed %d", m_maxBatch);
        }
        if (in.N != out.N)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Invalid input and output batch sizes: %d != %d", in.N, out.N);
        }
        if (in.uniqueFormat == NVCV_IMAGE_FORMAT_NONE || in.uniqueFormat != out.uniqueFormat)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT,
                          "Images in the input and output varshape must all have the same format");
        }
        FormatInfo fi = DecodeFormat(in.uniqueFormat);
        if (fi.planes != 1)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Images must have a single interleaved plane");
        }
        if (fi.channels > 4)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT, "Invalid channel number %d", fi.channels);
        }
        CheckBorder(border);
        NVCVTensorData dx;
        ExportTensor(hxform, dx, "Transformation matrix");
        const int  cols = m_perspective ? 9 : 6;
        DTypeInfo  dt   = DecodeDataType(dx.dtype);
        const bool ok   = dt.elem == kF32 && dt.channels == 1 && dx.rank == 2 && dx.shape[0] >= in.N
                     && dx.shape[1] == cols && dx.buffer.strided.strides[1] == 4;
        if (!ok)
        {
            throw OpError(NVCV_ERROR_INVALID_ARGUMENT,
                          "Transformation matrix tensor must be float32 of shape [N,%d] with packed rows, N >= %d", cols,
                          in.N);
        }
        WarpArgs a     = makeArgs(border, bval);
        a.srcList      = in.data.buffer.varShapeStrided.imageList;
        a.dstList      = out.data.buffer.varShapeStrided.imageList;
        a.xforms       = dx.buffer.strided.basePtr;
        a.xformStride  = dx.buffer.strided.strides[0];
        a.inverseGiven = (flags & NVCV_WARP_INVERSE_MAP) ? 1 : 0;
        DispatchType(fi.elem, fi.channels, flags & NVCV_INTERP_MAX, a, in.N, out.hostList, stream);
    }

private:
    WarpArgs makeArgs(NVCVBorderType border, float4 bval) const
    {
        WarpArgs a    = {};
        a.perspective = m_perspective ? 1 : 0;
        a.border      = (int32_t)border;
        a.bval[0]     = bval.x;
        a.bval[1]     = bval.y;
        a.bval[2]     = bval.z;
        a.bval[3]     = bval.w;
        return a;
    }

    bool    m_perspective;
    int32_t m_maxBatch;
};

class WarpAffine final : public Warp
{
public:
    explicit WarpAffine(int32_t maxBatch)
        : Warp(false, maxBatch)
    {
    }
};

class WarpPerspective final : public Warp
{
public:
    explicit WarpPerspective(int32_t maxBatch)
        : Warp(true, maxBatch)
    {
    }
};

} // namespace
} // namespace cvamd

using namespace cvamd;

extern "C"
{
CVCUDA_PUBLIC NVCVStatus cvcudaWarpAffineCreate(NVCVOperatorHandle *handle, const int32_t maxVarShapeBatchSize)
{
    return CreateOperator<WarpAffine>(handle, maxVarShapeBatchSize);
}

CVCUDA_PUBLIC NVCVStatus cvcudaWarpAffineSubmit(NVCVOperatorHandle handle, hipStream_t stream, NVCVTensorHandle in,
                                                NVCVTensorHandle out, const NVCVAffineTransform xform,
                                                const int32_t flags, const NVCVBorderType borderMode,
                                                const float4 borderValue)
{
    return Protect([&] { ToOperator<WarpAffine>(handle).submit(stream, in, out, xform, flags, borderMode, borderValue); });
}

CVCUDA_PUBLIC NVCVStatus cvcudaWarpAffineVarShapeSubmit(NVCVOperatorHandle handle, hipStream_t stream,
                                                        NVCVImageBatchHandle in, NVCVImageBatchHandle out,
                                                        NVCVTensorHandle transMatrix, const int32_t flags,
                                                        const NVCVBorderType borderMode, const float4 borderValue)
{
    return Protect(
        [&] { ToOperator<WarpAffine>(handle).submit(stream, in, out, transMatrix, flags, borderMode, borderValue); });
}

CVCUDA_PUBLIC NVCVStatus cvcudaWarpPerspectiveCreate(NVCVOperatorHandle *handle, const int32_t maxVarShapeBatchSize)
{
    return CreateOperator<WarpPerspective>(handle, maxVarShapeBatchSize);
}

CVCUDA_PUBLIC NVCVStatus cvcudaWarpPerspectiveSubmit(NVCVOperatorHandle handle, hipStream_t stream, NVCVTensorHandle in,
                                                     NVCVTensorHandle out, const NVCVPerspectiveTransform transMatrix,
                                                     const int32_t flags, const NVCVBorderType borderMode,
                                                     const float4 borderValue)
{
    return Protect(
        [&] { ToOperator<WarpPerspective>(handle).submit(stream, in, out, transMatrix, flags, borderMode, borderValue); });
}

CVCUDA_PUBLIC NVCVStatus cvcudaWarpPerspectiveVarShapeSubmit(NVCVOperatorHandle handle, hipStream_t stream,
                                                             NVCVImageBatchHandle in, NVCVImageBatchHandle out,
                                                             NVCVTensorHandle transMatrix, const int32_t flags,
                                                             const NVCVBorderType borderMode, const float4 borderValue)
{
    return Protect(
        [&]
        { ToOperator<WarpPerspective>(handle).submit(stream, in, out, transMatrix, flags, borderMode, borderValue); });
}
}

// What an image batch uploads, over a stand-in for the HIP runtime whose device memory is the host's: the lists on the device
// are those on the host after every export, and a batch with room for many more images than it holds does not copy that room.
// A batch that ends waits for its upload where the allocator of its lists does not.
#include <hip/hip_runtime_api.h>

#include <nvcv/Image.h>
#include <nvcv/ImageBatch.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

static int64_t g_copied = 0, g_copies = 0, g_waits = 0;

extern "C"
{
hipError_t hipMalloc(void **p, size_t n)
{
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    return hipMalloc(p, n);
}
hipError_t hipHostFree(void *p)
{
    return hipFree(p);
}
hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetLastError(void)
{
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t)
{
    return "";
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = reinterpret_cast<hipEvent_t>(1);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t)
{
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t)
{
    return hipSuccess;
}
hipError_t hipStreamGetDevice(hipStream_t stream, hipDevice_t *d)
{
    *d = stream == reinterpret_cast<hipStream_t>(0x1000) ? 1 : 0;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t)
{
    ++g_waits;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned)
{
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s)
{
    *s = hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(to, from, n);
    g_copied += (int64_t)n;
    ++g_copies;
    return hipSuccess;
}
}

#define REQUIRE(c)                                                                          \
    do                                                                                      \
    {                                                                                       \
        if (!(c))                                                                           \
        {                                                                                   \
            std::printf("line %d: %s (capacity %d)\n", __LINE__, #c, capacity);             \
            return 1;                                                                       \
        }                                                                                   \
    } while (0)

int main()
{
    const int64_t entry = sizeof(NVCVImageBufferStrided) + sizeof(NVCVImageFormat);
    for (int capacity : {3, 64, 5000, 1 << 20})
    {
        NVCVImageBatchVarShapeRequirements reqs;
        NVCVImageBatchHandle               batch = nullptr;
        REQUIRE(nvcvImageBatchVarShapeCalcRequirements(capacity, &reqs) == NVCV_SUCCESS);
        REQUIRE(nvcvImageBatchVarShapeConstruct(&reqs, nullptr, &batch) == NVCV_SUCCESS);
        int held = 0;
        for (int step = 0; step < 4; ++step)
        {
            if (step == 2)
            {
                REQUIRE(nvcvImageBatchVarShapeClear(batch) == NVCV_SUCCESS);
                held = 0;
            }
            NVCVImagePlaneStrided plane = {5 + step, 7, 256, reinterpret_cast<NVCVByte *>(uintptr_t(0x1000) * (step + 1))};
            REQUIRE(nvcvxImageBatchVarShapePushBuffers(batch, step % 2 ? NVCV_IMAGE_FORMAT_U8 : NVCV_IMAGE_FORMAT_RGB8, &plane, 1)
                    == NVCV_SUCCESS);
            ++held;
            g_copied = g_copies = 0;
            NVCVImageBatchData data;
            REQUIRE(nvcvImageBatchExportData(batch, nullptr, &data) == NVCV_SUCCESS);
            REQUIRE(g_copied >= entry && g_copied <= entry + 65536 && g_copies <= 2);
            REQUIRE(capacity > 64 || step % 2 || g_copies == 1); // a batch filled at once is one copy
            const NVCVImageBatchVarShapeBufferStrided &b = data.buffer.varShapeStrided;
            const NVCVImageBufferStrided              *host = nullptr;
            int32_t                                    n    = 0;
            REQUIRE(nvcvxImageBatchVarShapeGetHostImageList(batch, &host, &n) == NVCV_SUCCESS && n == held);
            REQUIRE(std::memcmp(b.imageList, host, n * sizeof(*host)) == 0);
            REQUIRE(std::memcmp(b.formatList, b.hostFormatList, n * sizeof(NVCVImageFormat)) == 0);
            REQUIRE(b.imageList[n - 1].planes[0].width == 5 + step && b.formatList[n - 1] == b.hostFormatList[n - 1]);
            g_copied = 0;
            REQUIRE(nvcvImageBatchExportData(batch, nullptr, &data) == NVCV_SUCCESS && g_copied == 0);
        }
        REQUIRE(nvcvImageBatchDecRef(batch, nullptr) == NVCV_SUCCESS);
    }
    // uploaded by its own device's stream, by another's, and by either with lists from the caller's own allocator
    for (int own = 0; own < 2; ++own)
    {
        for (uintptr_t stream : {uintptr_t(0), uintptr_t(0x2000), uintptr_t(0x1000)})
        {
            const int                          capacity = 4;
            NVCVImageBatchVarShapeRequirements reqs;
            NVCVImageBatchHandle               batch     = nullptr;
            NVCVAllocatorHandle                allocator = nullptr;
            NVCVResourceAllocator              host      = {};
            host.resType         = NVCV_RESOURCE_MEM_HOST_PINNED;
            host.res.mem.fnAlloc = [](void *, int64_t size, int32_t) { return std::malloc((size_t)size); };
            host.res.mem.fnFree  = [](void *, void *p, int64_t, int32_t) { std::free(p); };
            REQUIRE(own == 0 || nvcvAllocatorConstructCustom(&host, 1, &allocator) == NVCV_SUCCESS);
            REQUIRE(nvcvImageBatchVarShapeCalcRequirements(capacity, &reqs) == NVCV_SUCCESS);
            REQUIRE(nvcvImageBatchVarShapeConstruct(&reqs, allocator, &batch) == NVCV_SUCCESS);
            NVCVImagePlaneStrided plane = {5, 7, 256, reinterpret_cast<NVCVByte *>(0x1000)};
            REQUIRE(nvcvxImageBatchVarShapePushBuffers(batch, NVCV_IMAGE_FORMAT_U8, &plane, 1) == NVCV_SUCCESS);
            NVCVImageBatchData data;
            REQUIRE(nvcvImageBatchExportData(batch, reinterpret_cast<hipStream_t>(stream), &data) == NVCV_SUCCESS);
            g_waits = 0;
            REQUIRE(nvcvImageBatchDecRef(batch, nullptr) == NVCV_SUCCESS);
            REQUIRE((g_waits > 0) == (own == 1 || stream == 0x1000));
            REQUIRE(own == 0 || nvcvAllocatorDecRef(allocator, nullptr) == NVCV_SUCCESS);
        }
    }
    std::puts("ok");
    return 0;
}

/* A stand-in for the HIP runtime's entry points, preloaded so that the library plans and "launches"
 * on a host without a GPU: one device of 256 CUs and 160 KiB of LDS, allocations from the heap, kernels
 * that do nothing but leave their launch shape behind. */
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>
#include <stdlib.h>

static unsigned long long most_groups, most_threads, launches;

unsigned long long stub_most_groups(void) { return most_groups; }
unsigned long long stub_most_threads(void) { return most_threads; }
unsigned long long stub_launches(void) { return launches; }
void stub_reset(void) { most_groups = most_threads = launches = 0; }

hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int d) { (void)d; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d)
{
    (void)d;
    *v = a == hipDeviceAttributeMaxSharedMemoryPerBlock ? 160 * 1024 : a == hipDeviceAttributeMultiprocessorCount ? 256 : 0;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int d) { (void)p; (void)d; return hipErrorInvalidDevice; }
hipError_t hipRuntimeGetVersion(int *v) { *v = 0; return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n)
{
    *p = malloc(n ? n : 1);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
    (void)d; (void)s; (void)n; (void)k; (void)st;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f) { (void)f; *s = (hipStream_t)8; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *v)
{
    (void)s;
    *v = hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f) { (void)f; *e = (hipEvent_t)8; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { (void)e; (void)s; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned f) { (void)s; (void)e; (void)f; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute a, int v) { (void)f; (void)a; (void)v; return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t l)
{
    (void)f; (void)b; (void)l;
    *n = 2;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
/* the launch configuration between a call's <<<>>> and its stub */
static dim3 cfg_grid, cfg_block;
static size_t cfg_lds;
static hipStream_t cfg_stream;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s)
{
    cfg_grid = grid;
    cfg_block = block;
    cfg_lds = lds;
    cfg_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *s)
{
    *grid = cfg_grid;
    *block = cfg_block;
    *lds = cfg_lds;
    *s = cfg_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t lds, hipStream_t s)
{
    (void)f; (void)args; (void)lds; (void)s;
    const unsigned long long g = (unsigned long long)grid.x * grid.y * grid.z;
    ++launches;
    if (g > most_groups) most_groups = g;
    if (g * block.x > most_threads) most_threads = g * block.x;
    return hipSuccess;
}

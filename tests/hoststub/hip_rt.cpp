/*
 * hip_rt.cpp -- TEST INFRASTRUCTURE: a stand-in for the HIP runtime under the
 * host halves of the HIP sources (hipcc --offload-host-only), so that what a
 * launcher asks of the runtime is checked without a GPU: kernels do not run,
 * device memory is host memory, launches are held to the dynamic LDS size the
 * kernel was allowed.  One check per run:
 *   launch lds | slots
 */
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>

#include "jxamd.h"
extern "C" {
#include "jxamd_dev.h"
}

static const int LDS_LIMIT = 160 * 1024, LDS_DEFAULT = 64 * 1024;
static int mallocs, launches;
static hipError_t last, sync_error, stale; /* stale: another call's error, found by the next hipGetLastError */
static hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
static std::map<const void *, int> lds_allowed;
static std::function<void()> before_launch;
static void *arg6; /* the launch's seventh argument (the residual norm's work buffer) */

extern "C" {
hipError_t hipMalloc(void **p, size_t n) { mallocs++; *p = calloc(1, n ? n : 1); return hipSuccess; }
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetLastError(void)
{
    const hipError_t e = last != hipSuccess ? last : stale;
    last = stale = hipSuccess;
    return e;
}
hipError_t hipGetSymbolAddress(void **p, const void *)
{
    *p = calloc(1, 1 << 22);
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = LDS_LIMIT; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute a, int v)
{
    if (a == hipFuncAttributeMaxDynamicSharedMemorySize) lds_allowed[f] = v;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3 block, void **args, size_t shared, hipStream_t)
{
    if (before_launch) {
        std::function<void()> once;
        once.swap(before_launch);
        once();
    }
    const int allowed = lds_allowed.count(f) ? lds_allowed[f] : LDS_DEFAULT;
    if (shared > (size_t)allowed) return last = hipErrorInvalidValue;
    if (block.x == 256) arg6 = *(void **)args[6]; /* the kernels that clear have one thread, and one argument */
    launches++;
    return hipSuccess;
}
hipError_t hipLaunchCooperativeKernel(const void *, dim3, dim3, void **, unsigned int, hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return sync_error; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) { *s = capture; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *, unsigned int) { return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *, unsigned) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *, hipEvent_t, hipEvent_t) { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned int) { *p = calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned int) { *d = h; return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 2; return hipSuccess; }

static dim3 cfg_grid, cfg_block;
static size_t cfg_shared;
static hipStream_t cfg_stream;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st)
{
    cfg_grid = g; cfg_block = b; cfg_shared = s; cfg_stream = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *st)
{
    *g = cfg_grid; *b = cfg_block; *s = cfg_shared; *st = cfg_stream;
    return hipSuccess;
}
static void *handle;
void **__hipRegisterFatBinary(const void *) { return &handle; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned int, void *, void *, void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
}

static int fails;
#define CHECK(c) do { if (!(c)) { fails++; fprintf(stderr, "line %d: %s\n", __LINE__, #c); } } while (0)

static int gs_lds(int n, int xt)
{
    static const jxamd_lds_sweep sw = {nullptr, nullptr, nullptr, JXAMD_LDS_DEPTH};
    return jxamd_k_gs_lds(1, 4, 4, xt, n, &sw, &sw, nullptr, nullptr, 1, nullptr, 1, nullptr, nullptr, nullptr, nullptr);
}

/* a launch stays allowed whatever level another thread's handle sweeps between
 * its preparation and itself */
static void check_lds()
{
    const int xts[2] = {JXAMD_T_F64, JXAMD_T_F32};
    for (int xt : xts) {
        const int most = jxamd_gs_lds_rows(xt);
        CHECK(most > 16384 && gs_lds(most, xt) == 0 && gs_lds(most + 1, xt) == JXAMD_ERROR_ARG);
        for (int small : {1, 9000, most - 1}) {
            before_launch = [=] { CHECK(gs_lds(small, xt) == 0); };
            CHECK(gs_lds(most, xt) == 0);
            CHECK(!before_launch);
        }
    }
}

static int norm()
{
    static int ia[2] = {0, 1}, ja[1];
    static double a[4], x[2], b[2], o[2];
    return jxamd_bsr_residual_norm(1, 2, ia, ja, a, x, b, o, nullptr);
}

/* the residual norm's work buffers in the module: given back whenever no
 * launch can still use them, whatever the call returns */
static void check_slots()
{
    CHECK(norm() == 0 && mallocs == 0);
    const void *first = arg6;
    for (int k = 0; k < 20; k++) {
        stale = hipErrorInvalidValue; /* of an earlier call: reported, but the launch was made and has ended */
        CHECK(norm() == JXAMD_ERROR_DEVICE);
    }
    CHECK(norm() == 0 && mallocs == 0);
    /* a stream being captured: the wait is refused, and the call's memory is its own */
    capture = hipStreamCaptureStatusActive;
    sync_error = hipErrorStreamCaptureUnsupported;
    for (int k = 0; k < 20; k++) CHECK(norm() == JXAMD_ERROR_DEVICE && mallocs == k + 1);
    capture = hipStreamCaptureStatusNone;
    sync_error = hipSuccess;
    CHECK(norm() == 0 && mallocs == 20 && arg6 == first);
    /* a wait that fails: the launch may still run, its buffer is not handed out again */
    sync_error = hipErrorUnknown;
    CHECK(norm() == JXAMD_ERROR_DEVICE && arg6 == first);
    sync_error = hipSuccess;
    CHECK(norm() == 0 && mallocs == 20 && arg6 != first);
}

int main(int argc, char **argv)
{
    if (argc == 2 && !strcmp(argv[1], "lds")) check_lds();
    else if (argc == 2 && !strcmp(argv[1], "slots")) check_slots();
    else return 2;
    printf("launches %d mallocs %d fails %d\n", launches, mallocs, fails);
    return fails ? 1 : 0;
}

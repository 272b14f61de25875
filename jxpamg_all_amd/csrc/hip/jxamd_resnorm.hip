// jxamd_resnorm.hip -- true residual norm of a BSR system on the device.
//
// norms[0] = ||b - A x||_2, norms[1] = ||b||_2 for A in the reference's BSR
// layout (0-based ia[nb+1], ja[nnzb], row-major b x b blocks), in one launch:
// each thread owns scalar rows (i, r) on a grid-stride loop and accumulates
// the squares of r_(i,r) = b_(i,r) - sum_k A_k[r][:] x_(ja[k]), workgroup
// partials go to a scratch array, and the last workgroup to finish adds them
// in a fixed order, so the result does not depend on scheduling.
//
// This is the check GMRES makes on convergence (the reference copies b, runs
// its matvec with alpha = -1, beta = 1 and takes the square root of the inner
// product: jxfpamg-0220/csrc/krylov/pgmres.c:1505-1511; ||b|| as at
// pgmres.c:1062).
#include <hip/hip_runtime.h>

#include <mutex>

extern "C" {
#include "jxamd_dev.h"
}

#define RN_THREADS 256
#define RN_WAVE 64
// the grid never exceeds RN_MAX_GROUPS workgroups (grid-stride loop), so a
// work buffer of RN_SCRATCH_BYTES always holds every partial
#define RN_MAX_GROUPS 2048
// work buffer layout: double partials[2 * RN_MAX_GROUPS], then the arrival counter
#define RN_PART_BYTES (2 * RN_MAX_GROUPS * sizeof(double))
#define RN_SCRATCH_BYTES (RN_PART_BYTES + 256)

namespace {

// One scalar row per lane: the B lanes of a block row read the rows of a block
// side by side.  U blocks' columns, then their values and x, are loaded before
// the first is used (a row's loop had one chain of two dependent trips in flight
// per block: 75x81x67 4x4 87 us, 81 now).  VEC: a and x on 16-byte boundaries,
// B even: pairs in one load.
template <int B, int U, bool VEC>
__global__ void __launch_bounds__(RN_THREADS) k_bsr_resnorm(int nb, const int *__restrict__ ia,
                                                            const int *__restrict__ ja,
                                                            const double *__restrict__ a,
                                                            const double *__restrict__ x,
                                                            const double *__restrict__ bv, double *part,
                                                            unsigned int *count, double *norms)
{
    __shared__ double sr[RN_THREADS / RN_WAVE], sb[RN_THREADS / RN_WAVE];
    __shared__ bool last;
    const long long n = (long long)nb * B;
    double rr = 0.0, bb = 0.0;
    for (long long row = (long long)blockIdx.x * RN_THREADS + threadIdx.x; row < n;
         row += (long long)gridDim.x * RN_THREADS) {
        const int i = (int)(row / B), r = (int)(row % B);
        const double bi = bv[row];
        double s = bi;
        const int k1 = ia[i + 1];
        for (int k = ia[i]; k < k1; k += U) {
            int j[U];
            double av[U][B], xv[U][B];
#pragma unroll
            for (int u = 0; u < U; u++) j[u] = ja[min(k + u, k1 - 1)];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const double *blk = a + (size_t)min(k + u, k1 - 1) * (B * B) + r * B;
                const double *xj = x + (size_t)j[u] * B;
                if constexpr (VEC) {
                    typedef double __attribute__((ext_vector_type(2))) D2;
#pragma unroll
                    for (int c = 0; c < B; c += 2) {
                        const D2 a2 = *reinterpret_cast<const D2 *>(blk + c), x2 = *reinterpret_cast<const D2 *>(xj + c);
                        av[u][c] = a2[0];
                        av[u][c + 1] = a2[1];
                        xv[u][c] = x2[0];
                        xv[u][c + 1] = x2[1];
                    }
                } else {
#pragma unroll
                    for (int c = 0; c < B; c++) {
                        av[u][c] = blk[c];
                        xv[u][c] = xj[c];
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (k + u < k1)
#pragma unroll
                    for (int c = 0; c < B; c++) s -= av[u][c] * xv[u][c];
        }
        rr += s * s;
        bb += bi * bi;
    }
#pragma unroll
    for (int off = RN_WAVE / 2; off > 0; off >>= 1) {
        rr += __shfl_xor(rr, off);
        bb += __shfl_xor(bb, off);
    }
    if (threadIdx.x % RN_WAVE == 0) {
        sr[threadIdx.x / RN_WAVE] = rr;
        sb[threadIdx.x / RN_WAVE] = bb;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double r0 = 0.0, b0 = 0.0;
        for (int w = 0; w < RN_THREADS / RN_WAVE; w++) {
            r0 += sr[w];
            b0 += sb[w];
        }
        // device-scope stores of the partials, completed before the arrival
        // is counted; the last arrival reads them with device-scope loads
        __hip_atomic_store(part + 2 * blockIdx.x, r0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(part + 2 * blockIdx.x + 1, b0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_waitcnt(0);
        const unsigned int prev = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = (prev == gridDim.x - 1);
    }
    __syncthreads();
    if (!last) return;
    // fixed-order sum over the partials: thread t adds partials t, t + 256, ...
    rr = 0.0;
    bb = 0.0;
    for (unsigned int g = threadIdx.x; g < gridDim.x; g += RN_THREADS) {
        rr += __hip_atomic_load(part + 2 * g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        bb += __hip_atomic_load(part + 2 * g + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int off = RN_WAVE / 2; off > 0; off >>= 1) {
        rr += __shfl_xor(rr, off);
        bb += __shfl_xor(bb, off);
    }
    __syncthreads();
    if (threadIdx.x % RN_WAVE == 0) {
        sr[threadIdx.x / RN_WAVE] = rr;
        sb[threadIdx.x / RN_WAVE] = bb;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double r0 = 0.0, b0 = 0.0;
        for (int w = 0; w < RN_THREADS / RN_WAVE; w++) {
            r0 += sr[w];
            b0 += sb[w];
        }
        norms[0] = sqrt(r0);
        norms[1] = sqrt(b0);
        __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

__global__ void k_rn_clear(unsigned int *count) { *count = 0u; }

int rn_check(int nb, int b, const int *ia, const int *ja, const double *a, const double *x, const double *bv,
             double *norms)
{
    if (nb < 0 || b < 1 || b > JXAMD_MAX_BLOCK || !norms) return JXAMD_ERROR_ARG;
    if (nb > 0 && (!ia || !ja || !a || !x || !bv)) return JXAMD_ERROR_ARG;
    // scalar rows are counted in 64-bit, block rows and block positions in int32
    if ((long long)nb * b > (long long)0x7fffffff) return JXAMD_ERROR_ARG;
    return 0;
}

int rn_grid(int nb, int b)
{
    const long long n = (long long)nb * b;
    long long g = (n + RN_THREADS - 1) / RN_THREADS;
    if (g < 1) g = 1;
    if (g > RN_MAX_GROUPS) g = RN_MAX_GROUPS;
    return (int)g;
}

int rn_launch(int nb, int b, const int *ia, const int *ja, const double *a, const double *x, const double *bv,
              double *norms, double *part, unsigned int *count, bool clear, hipStream_t st)
{
    const int grid = rn_grid(nb, b);
    if (grid > RN_MAX_GROUPS) return JXAMD_ERROR_ARG;
    if (clear) hipLaunchKernelGGL(k_rn_clear, dim3(1), dim3(1), 0, st, count);
    const bool vec = ((uintptr_t)a | (uintptr_t)x) % 16 == 0;
#define RN_LAUNCH(BS, US, VS)                                                                                          \
    hipLaunchKernelGGL((k_bsr_resnorm<BS, US, VS>), dim3(grid), dim3(RN_THREADS), 0, st, nb, ia, ja, a, x, bv, part,   \
                       count, norms)
    switch (b) {
    case 1: RN_LAUNCH(1, 8, false); break;
    case 2:
        if (vec) RN_LAUNCH(2, 8, true);
        else RN_LAUNCH(2, 8, false);
        break;
    case 3: RN_LAUNCH(3, 4, false); break;
    default:
        if (vec) RN_LAUNCH(4, 4, true);
        else RN_LAUNCH(4, 4, false);
        break;
    }
#undef RN_LAUNCH
    return hipGetLastError() == hipSuccess ? 0 : JXAMD_ERROR_DEVICE;
}

// Scratch of the allocation-free entry point.  In host code `scratch` names
// a host-side stand-in, not device memory: only the address returned by
// hipGetSymbolAddress (one per device) may be handed to kernels.
static __device__ __align__(256) unsigned char scratch[RN_SCRATCH_BYTES];

#define RN_MAX_DEVICES 64
std::mutex rn_mutex;
void *rn_scratch_dev[RN_MAX_DEVICES];

// this device's copy of the scratch array, looked up once per device
int rn_scratch(void **out)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return JXAMD_ERROR_DEVICE;
    if (dev < 0 || dev >= RN_MAX_DEVICES) return JXAMD_ERROR_DEVICE;
    std::lock_guard<std::mutex> g(rn_mutex);
    if (!rn_scratch_dev[dev]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return JXAMD_ERROR_DEVICE;
        rn_scratch_dev[dev] = p;
    }
    *out = rn_scratch_dev[dev];
    return 0;
}

// Work buffers of the entry point that waits for its result: one of RN_SLOTS
// in the module's own memory for the call's duration (with an allocation and a
// release per call, and the launch that clears a fresh counter, a call took
// 5 us longer); a call that finds none free allocates its own, and so does one
// on a stream that is being captured, whose launch might run after the call.
#define RN_SLOTS 8
static __device__ __align__(256) unsigned char slots[RN_SLOTS * RN_SCRATCH_BYTES];
void *rn_slots_dev[RN_MAX_DEVICES];
unsigned int rn_slots_used[RN_MAX_DEVICES]; // bit k: slot k, under rn_mutex

// a free slot of this device: its number and address, or -1
int rn_slot_take(hipStream_t st, int *dev, void **out)
{
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) return -1;
    if (hipGetDevice(dev) != hipSuccess || *dev < 0 || *dev >= RN_MAX_DEVICES) return -1;
    std::lock_guard<std::mutex> g(rn_mutex);
    if (!rn_slots_dev[*dev]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(slots)) != hipSuccess || !p) return -1;
        rn_slots_dev[*dev] = p;
    }
    for (int k = 0; k < RN_SLOTS; k++)
        if (!(rn_slots_used[*dev] >> k & 1u)) {
            rn_slots_used[*dev] |= 1u << k;
            *out = (unsigned char *)rn_slots_dev[*dev] + (size_t)k * RN_SCRATCH_BYTES;
            return k;
        }
    return -1;
}
void rn_slot_give(int dev, int k)
{
    std::lock_guard<std::mutex> g(rn_mutex);
    rn_slots_used[dev] &= ~(1u << k);
}

} // namespace

extern "C" {

int jxamd_bsr_residual_norm(int nb, int b, const int *d_ia, const int *d_ja, const double *d_a, const double *d_x,
                            const double *d_b, double *d_norms, void *stream)
{
    int e = rn_check(nb, b, d_ia, d_ja, d_a, d_x, d_b, d_norms);
    if (e) return e;
    hipStream_t st = (hipStream_t)stream;
    void *work = nullptr;
    int dev = 0;
    const int slot = rn_slot_take(st, &dev, &work);
    if (slot < 0 && hipMalloc(&work, RN_SCRATCH_BYTES) != hipSuccess) return JXAMD_ERROR_MEMORY;
    // a slot's counter is zero: at first, and again after every finished launch
    e = rn_launch(nb, b, d_ia, d_ja, d_a, d_x, d_b, d_norms, (double *)work,
                  (unsigned int *)((unsigned char *)work + RN_PART_BYTES), slot < 0, st);
    // the launch must finish before its partials are released
    const bool ended = hipStreamSynchronize(st) == hipSuccess;
    if (!ended && !e) e = JXAMD_ERROR_DEVICE;
    if (slot >= 0) {
        // whatever the launch reported; where the wait failed, it may not have
        // run to its end and the slot stays out of use
        if (ended) rn_slot_give(dev, slot);
    } else if (hipFree(work) != hipSuccess && !e) {
        e = JXAMD_ERROR_DEVICE;
    }
    return e;
}

int jxamd_bsr_residual_norm_noalloc(int nb, int b, const int *d_ia, const int *d_ja, const double *d_a,
                                    const double *d_x, const double *d_b, double *d_norms, void *stream)
{
    int e = rn_check(nb, b, d_ia, d_ja, d_a, d_x, d_b, d_norms);
    if (e) return e;
    void *work = nullptr;
    e = rn_scratch(&work);
    if (e) return e;
    return rn_launch(nb, b, d_ia, d_ja, d_a, d_x, d_b, d_norms, (double *)work,
                     (unsigned int *)((unsigned char *)work + RN_PART_BYTES), true, (hipStream_t)stream);
}

} // extern "C"

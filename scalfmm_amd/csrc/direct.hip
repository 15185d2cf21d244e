// direct.hip -- FP64 direct summation on the device for sampled targets: the
// O(N^2) reference the FMM results are measured against, as the reference's
// test programs compute it pair by pair with FP2P::NonMutualParticles
// (Tests/Kernels/DirectAlgorithm.cpp:203-215, Src/Kernels/P2P/FP2P.hpp:80-101).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <string>

#include "fmm_common.hpp"
#include "hfmm_internal.hpp"

namespace hfmm {
namespace {

constexpr int kDirectBlock = 256;
constexpr int kDirectTargets = 8;  // targets per workgroup (sources are read once for all of them)

// A workgroup per kDirectTargets targets and share of the sources: the threads
// stride over the share, then a tree reduction in LDS per target.  Force
// convention F = q_t * sum_j -q_j d / r^3, the FMM's.  With several shares the
// sums go to part[share][4][nt] and k_direct_sum adds them in order.  One
// share per target group left 3,001 targets to 376 workgroups (1.4 per CU) and
// one target to a single one.
__global__ __launch_bounds__(kDirectBlock) void k_direct(int64_t n, const double* __restrict__ x,
                                                        const double* __restrict__ y, const double* __restrict__ z,
                                                        const double* __restrict__ q,
                                                        const int64_t* __restrict__ targets, int64_t nt,
                                                        double* __restrict__ out, double* __restrict__ part) {
    __shared__ double red[4][kDirectBlock];
    int64_t t[kDirectTargets];
    double tx[kDirectTargets], ty[kDirectTargets], tz[kDirectTargets], acc[kDirectTargets][4];
#pragma unroll
    for (int u = 0; u < kDirectTargets; ++u) {
        const int64_t g = static_cast<int64_t>(blockIdx.x) * kDirectTargets + u;
        t[u] = g < nt ? targets[g] : -1;
        const int64_t tt = t[u] >= 0 ? t[u] : 0;
        tx[u] = x[tt];
        ty[u] = y[tt];
        tz[u] = z[tt];
        for (int k = 0; k < 4; ++k) acc[u][k] = 0.;
    }
    const int64_t j0 = n * blockIdx.y / gridDim.y, j1 = n * (blockIdx.y + 1) / gridDim.y;
    for (int64_t j = j0 + threadIdx.x; j < j1; j += kDirectBlock) {
        const double xj = x[j], yj = y[j], zj = z[j], qj = q[j];
#pragma unroll
        for (int u = 0; u < kDirectTargets; ++u) {
            const double dx = tx[u] - xj, dy = ty[u] - yj, dz = tz[u] - zj;
            double inv = rsqrt_f64_any(dx * dx + dy * dy + dz * dz);
            const double q1 = j == t[u] ? 0. : qj;
            inv = j == t[u] ? 0. : inv;
            const double qi = q1 * inv;
            const double qi3 = qi * inv * inv;
            acc[u][0] += qi;
            acc[u][1] -= qi3 * dx;
            acc[u][2] -= qi3 * dy;
            acc[u][3] -= qi3 * dz;
        }
    }
    for (int u = 0; u < kDirectTargets; ++u) {
        for (int k = 0; k < 4; ++k) red[k][threadIdx.x] = acc[u][k];
        __syncthreads();
        for (int s = kDirectBlock / 2; s > 0; s >>= 1) {
            if (threadIdx.x < s)
                for (int k = 0; k < 4; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + s];
            __syncthreads();
        }
        if (threadIdx.x == 0 && t[u] >= 0) {
            const int64_t g = static_cast<int64_t>(blockIdx.x) * kDirectTargets + u;
            if (gridDim.y > 1) {
                for (int k = 0; k < 4; ++k) part[(blockIdx.y * 4 + k) * nt + g] = red[k][0];
            } else {
                const double qt = q[t[u]];
                out[g] = red[0][0];
                out[nt + g] = red[1][0] * qt;
                out[2 * nt + g] = red[2][0] * qt;
                out[3 * nt + g] = red[3][0] * qt;
            }
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(kDirectBlock) void k_direct_sum(const double* __restrict__ q,
                                                            const int64_t* __restrict__ targets, int64_t nt, int shares,
                                                            const double* __restrict__ part, double* __restrict__ out) {
    const int64_t g = static_cast<int64_t>(blockIdx.x) * kDirectBlock + threadIdx.x;
    if (g >= nt) return;
    // compensated (each addition's exact error is carried along): dozens of plain
    // additions cost the last digit of sums whose terms have one sign
    double s[4] = {0., 0., 0., 0.}, e[4] = {0., 0., 0., 0.};
    for (int i = 0; i < shares; ++i)
        for (int k = 0; k < 4; ++k) {
            const double v = part[(static_cast<int64_t>(i) * 4 + k) * nt + g], t = s[k] + v, w = t - s[k];
            e[k] += (s[k] - (t - w)) + (v - w);
            s[k] = t;
        }
    // a sum that left the finite numbers stands as it is
    for (int k = 0; k < 4; ++k) s[k] = isfinite(s[k]) ? s[k] + e[k] : s[k];
    const double qt = q[targets[g]];
    out[g] = s[0];
    for (int k = 1; k < 4; ++k) out[k * nt + g] = s[k] * qt;
}

// Staging of hfmm_direct_noalloc: the target indices (kDirectStaticTargets
// int64) followed by the results (4 kDirectStaticTargets doubles), 40 bytes per
// target, 2.5 MiB in all.  Every GPU the library runs on holds its own copy
// until the process ends; host code uses the per-device address that
// init_direct_scratch reads, never the array's name.
constexpr int64_t kDirectStaticTargets = HFMM_DIRECT_NOALLOC_MAX_TARGETS;
__device__ __align__(256) unsigned char scratch[kDirectStaticTargets * 5 * sizeof(double)];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};  // device address of `scratch` per device

// Shares of the sources: enough for kDirectBlocks workgroups, a round of the
// threads or more each, partial sums (32 bytes per target and share) within the
// static staging beside the 40 bytes per target, so that both entry points
// split, and sum, alike.
constexpr int64_t kDirectBlocks = 2048;

int direct_shares(int64_t n, int64_t nt) {
    const int64_t blocks = (nt + kDirectTargets - 1) / kDirectTargets;
    int64_t s = (kDirectBlocks + blocks - 1) / blocks;
    s = std::min(s, (n + kDirectBlock - 1) / kDirectBlock);
    s = std::min<int64_t>(s, (kDirectStaticTargets * 40 - nt * 40) / (nt * 32));
    return static_cast<int>(std::max<int64_t>(1, s));
}

// Launch of k_direct over c's particles for nt targets whose indices are at
// device address dt, results (four arrays of nt) at dout, followed by room for
// the partial sums of direct_shares.
int launch_direct(Context* c, int64_t nt, const int64_t* dt, double* dout) {
    const int64_t blocks = (nt + kDirectTargets - 1) / kDirectTargets;
    const int shares = direct_shares(c->n, nt);
    double* part = dout + 4 * nt;
    hipLaunchKernelGGL(k_direct, dim3(static_cast<unsigned>(blocks), static_cast<unsigned>(shares)), dim3(kDirectBlock), 0,
                       c->stream, c->n, c->x, c->y, c->z, c->q, dt, nt, dout, part);
    HFMM_TRY(check_launch(c, "direct"));
    if (shares == 1) return HFMM_OK;
    hipLaunchKernelGGL(k_direct_sum, dim3(static_cast<unsigned>((nt + kDirectBlock - 1) / kDirectBlock)),
                       dim3(kDirectBlock), 0, c->stream, c->q, dt, nt, shares, part, dout);
    return check_launch(c, "direct_sum");
}

// Copies the four result arrays at dout (nt each) into the caller's host
// arrays (NULL skips one) and waits for them.
int copy_direct_results(Context* c, int64_t nt, const double* dout, double* pot, double* fx, double* fy, double* fz) {
    double* outs[4] = {pot, fx, fy, fz};
    for (int k = 0; k < 4; ++k)
        if (outs[k] && hipMemcpyAsync(outs[k], dout + k * nt, sizeof(double) * nt, hipMemcpyDeviceToHost, c->stream) !=
                           hipSuccess)
            return fail(c, HFMM_ERR_DEVICE, "direct: result copy failed");
    if (hipStreamSynchronize(c->stream) != hipSuccess) return fail(c, HFMM_ERR_DEVICE, "direct: synchronize failed");
    return HFMM_OK;
}

}  // namespace

int init_direct_scratch(Context* c) {
    if (c->device < 0 || c->device >= kMaxDevices) return fail(c, HFMM_ERR_ARG, "direct staging: device index too large");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[c->device]) return HFMM_OK;
    if (hipSetDevice(c->device) != hipSuccess) return fail(c, HFMM_ERR_DEVICE, "direct staging: hipSetDevice failed");
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
        return fail(c, HFMM_ERR_DEVICE, std::string("direct staging: hipGetSymbolAddress failed: ") + hipGetErrorString(e));
    g_scratch_ptr[c->device] = ptr;
    return HFMM_OK;
}

int direct_sum_noalloc(Context* c, int64_t nt, const int64_t* targets, double* pot, double* fx, double* fy,
                       double* fz) {
    if (nt > kDirectStaticTargets)
        return fail(c, HFMM_ERR_ARG,
                    "direct_noalloc: " + std::to_string(nt) + " targets exceed the static staging's " +
                        std::to_string(kDirectStaticTargets));
    void* base = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        if (c->device >= 0 && c->device < kMaxDevices) base = g_scratch_ptr[c->device];
    }
    if (!base) return fail(c, HFMM_ERR_STATE, "direct_noalloc: the static staging of this device is not set up");
    int64_t* dt = static_cast<int64_t*>(base);
    double* dout = reinterpret_cast<double*>(dt + nt);
    // every call rewrites the staging it reads: the target indices here, each
    // result entry by the kernel (one per target), so nothing needs clearing
    if (hipMemcpyAsync(dt, targets, sizeof(int64_t) * nt, hipMemcpyHostToDevice, c->stream) != hipSuccess)
        return fail(c, HFMM_ERR_DEVICE, "direct_noalloc: target copy failed");
    HFMM_TRY(launch_direct(c, nt, dt, dout));
    return copy_direct_results(c, nt, dout, pot, fx, fy, fz);
}

int direct_sum(Context* c, int64_t nt, const int64_t* targets, double* pot, double* fx, double* fy, double* fz) {
    // staging kept by the context: indices, results, partial sums
    HFMM_TRY(ensure(c, c->d_direct, static_cast<size_t>(nt) * (40 + 32 * direct_shares(c->n, nt))));
    int64_t* dt = c->d_direct.as<int64_t>();
    double* dout = reinterpret_cast<double*>(dt + nt);
    if (hipMemcpyAsync(dt, targets, sizeof(int64_t) * nt, hipMemcpyHostToDevice, c->stream) != hipSuccess)
        return fail(c, HFMM_ERR_DEVICE, "direct: target copy failed");
    HFMM_TRY(launch_direct(c, nt, dt, dout));
    return copy_direct_results(c, nt, dout, pot, fx, fy, fz);
}

}  // namespace hfmm

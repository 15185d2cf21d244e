// fmm_device.hip -- FP64 FMM passes of the Chebyshev 1/r kernel on CDNA4.
//
//   P2M  per leaf: M_n += sum_p q_p Sx(xi_p, n_x) Sy(.., n_y) Sz(.., n_z)
//        (Src/Kernels/Chebyshev/FChebInterpolator.hpp:625-762)
//   M2M  per parent: three 1-D contractions per child (FChebInterpolator.hpp:560-584)
//   M2L  m2l_f64.hip
//   L2L  per parent: transposed contractions (FChebInterpolator.hpp:587-611)
//   L2P  per leaf: potential and q * gradient (FChebInterpolator.hpp:1220-1417)
//   P2P  per target particle over the 27-leaf neighbourhood
//        (Src/Kernels/P2P/FP2P.hpp:103-269 conventions)
#include <hip/hip_runtime.h>

#include <algorithm>

#include "fmm_common.hpp"
#include "hfmm_internal.hpp"

namespace hfmm {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

// S(xi, root_j) = 1/p + 2/p sum_{o>=1} T_o(xi) T_o(root_j); dS = d/dxi S.
template <int P, bool GRAD>
__device__ __forceinline__ void interp_weights(double xi, const double* __restrict__ sT, double* S, double* dS) {
    double T[P], U[P];
    T[0] = 1.;
    if (P > 1) T[1] = xi;
    U[0] = 1.;
    if (P > 1) U[1] = 2. * xi;
#pragma unroll
    for (int j = 2; j < P; ++j) {
        T[j] = 2. * xi * T[j - 1] - T[j - 2];
        if (GRAD) U[j] = 2. * xi * U[j - 1] - U[j - 2];
    }
#pragma unroll
    for (int j = 0; j < P; ++j) {
        double s = 1. / P, ds = 0.;
#pragma unroll
        for (int o = 1; o < P; ++o) {
            const double t = sT[o * P + j];
            s += 2. / P * T[o] * t;
            if (GRAD) ds += 2. / P * (o * U[o - 1]) * t;
        }
        S[j] = s;
        if (GRAD) dS[j] = ds;
    }
}

constexpr int kUniformMaxOrder = 8;  // the uniform scheme's dense M2L holds p^3 <= 512 ranks

// FUnifRoots::L and ::dL (Src/Kernels/Uniform/FUnifRoots.hpp:49-118) on the
// equispaced roots r: L_n by the scaled product, dL_n by the sum of products
// over the root table; the argument clamped to [-1, 1].
template <int P, bool GRAD>
__device__ __forceinline__ void lagrange_weights(double xi, const double* __restrict__ r, double* S, double* dS) {
    const double x = fmin(fmax(xi, -1.), 1.);
#pragma unroll
    for (int n = 0; n < P; ++n) {
        const int omn = P - n - 1;
        double fn = 1., fo = 1.;
        for (int i = 2; i <= n; ++i) fn *= i;
        for (int i = 2; i <= omn; ++i) fo *= i;
        double scale = (omn % 2) ? -1. : 1.;
        double p2 = 1.;
        for (int i = 0; i < P - 1; ++i) p2 *= 2.;
        scale /= p2 * fn * fo;
        double L = 1.;
#pragma unroll
        for (int m = 0; m < P; ++m)
            if (m != n) L *= static_cast<double>(P - 1) * (x + 1.) - 2. * m;
        S[n] = L * scale;
        if (GRAD) {
            double num = 0., den = 1.;
#pragma unroll
            for (int q = 0; q < P; ++q) {
                if (q == n) continue;
                double t = 1.;
#pragma unroll
                for (int m = 0; m < P; ++m)
                    if (m != n && m != q) t *= x - r[m];
                num += t;
                den *= r[n] - r[q];
            }
            dS[n] = num / den;
        }
    }
}

// ---------------------------------------------------------------------------
// P2M: one wave per window of 64 sorted particles.  Each lane forms the
// interpolation weights of its particle in the LDS; the wave then walks the
// leaves that start in the window, lanes over the coefficients.  A leaf that
// ends inside the window sums its particles from the LDS in one round (most
// leaves hold a few particles); the last leaf of a window may run past it and
// is summed in rounds of 64 particles from its first one.  A leaf's rounds
// always begin at its first particle, so its sums do not depend on where the
// windows fall.
template <int P, int BASIS>
__device__ __forceinline__ void p2m_weights(const double* __restrict__ sp, int64_t n, int64_t e, Box bx,
                                            uint64_t lkey, const double* __restrict__ sT,
                                            const double* __restrict__ uroots, double* S, double* Q) {
    double a[3], b[3];
    leaf_bounds(bx, lkey, a, b);
    const double pos[3] = {sp[e], sp[n + e], sp[2 * n + e]};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const double xi = (2. * pos[d] - b[d] - a[d]) / (b[d] - a[d]);
        if constexpr (BASIS == 1)
            lagrange_weights<P, false>(xi, uroots, S + d * P, nullptr);
        else
            interp_weights<P, false>(xi, sT, S + d * P, nullptr);
    }
    *Q = sp[3 * n + e];
}

template <int P, int BASIS>
__global__ __launch_bounds__(64) void k_p2m(int64_t n, const int32_t* __restrict__ pleaf,
                                           const uint64_t* __restrict__ lkeys, const int32_t* __restrict__ lstart,
                                           const double* __restrict__ sp, Box bx, const double* __restrict__ Troots,
                                           const double* __restrict__ uroots, double* __restrict__ M, int LD) {
    constexpr int NN = P * P * P;
    constexpr int PER = (NN + 63) / 64;
    __shared__ double sS[64][3 * P];
    __shared__ double sQ[64];
    __shared__ double sT[P * P];
    __shared__ int sStart[65];
    const int lane = threadIdx.x;
    const int64_t w0 = static_cast<int64_t>(blockIdx.x) * 64;
    const int64_t wend = min(w0 + 64, n);
    for (int i = lane; i < P * P; i += 64) sT[i] = Troots[i];
    // the leaves that start in the window: first .. last
    int first = pleaf[w0];
    if (lstart[first] < w0) ++first;
    const int last = pleaf[wend - 1];
    if (first > last) return;  // inside one long leaf: its first window sums it
    __syncthreads();
    if (w0 + lane < wend) p2m_weights<P, BASIS>(sp, n, w0 + lane, bx, lkeys[pleaf[w0 + lane]], sT, uroots,
                                                &sS[lane][0], &sQ[lane]);
    // the bounds of the window's leaves (at most 64) through the LDS: the leaf
    // loop then holds no vector load, whose wait would also cover the stores
    // of the previous leaves
    if (lane <= last - first) sStart[lane] = lstart[first + lane];
    if (lane == 0) sStart[last - first + 1] = lstart[last + 1];
    __syncthreads();
    for (int leaf = first; leaf <= last; ++leaf) {
        const int s0 = sStart[leaf - first], s1 = sStart[leaf - first + 1];
        double acc[PER];
#pragma unroll
        for (int t = 0; t < PER; ++t) acc[t] = 0.;
        // one round over particles m0 .. m1-1 of the LDS rows; per coefficient the
        // terms are added in particle order
        auto round = [&](int m0, int m1) {
            double sum[PER];
#pragma unroll
            for (int t = 0; t < PER; ++t) sum[t] = 0.;
            for (int m = m0; m < m1; ++m) {
                const double q = sQ[m];
#pragma unroll
                for (int t = 0; t < PER; ++t) {
                    const int idx = lane + 64 * t;
                    const int i = idx % P, j = (idx / P) % P, k = idx / (P * P);
                    if (NN % 64 == 0 || idx < NN) sum[t] += q * sS[m][P + j] * sS[m][2 * P + k] * sS[m][i];
                }
            }
#pragma unroll
            for (int t = 0; t < PER; ++t) acc[t] += sum[t];
        };
        if (s1 <= wend) {
            round(static_cast<int>(s0 - w0), static_cast<int>(s1 - w0));
        } else {
            // the window's last leaf runs past it: rounds of 64 from s0
            for (int base = s0; base < s1; base += 64) {
                const int cnt = min(64, s1 - base);
                __syncthreads();
                if (lane < cnt)
                    p2m_weights<P, BASIS>(sp, n, base + lane, bx, lkeys[leaf], sT, uroots, &sS[lane][0], &sQ[lane]);
                __syncthreads();
                round(0, cnt);
            }
        }
#pragma unroll
        for (int t = 0; t < PER; ++t) {
            const int idx = lane + 64 * t;
            if (idx < LD) M[static_cast<int64_t>(leaf) * LD + idx] = idx < NN ? acc[t] : 0.;  // zero padding
        }
    }
}

// ---------------------------------------------------------------------------
// M2M and L2L: a workgroup of 4 waves shares the 8 children's interpolation
// matrices in the LDS, one parent per wave.  The waves of a workgroup walk
// different numbers of children, so the separable passes through each wave's
// own LDS buffers are ordered by wave-local fences: the wave's LDS accesses run
// in order, and the fence keeps the compiler from moving other lanes' reads
// above the writes they depend on.
__device__ __forceinline__ void wave_lds_order() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront"); }

// M2M: child[m] -> parent[n] += Sx[nx][mx] Sy[ny][my] Sz[nz][mz] child[m].
template <int P>
__global__ __launch_bounds__(256) void k_m2m(int np, const int32_t* __restrict__ cstart,
                                            const uint64_t* __restrict__ ckeys, const double* __restrict__ interp,
                                            const double* __restrict__ Mc, double* __restrict__ Mp, int LD) {
    constexpr int NN = P * P * P;
    constexpr int PER = (NN + 63) / 64;
    __shared__ double sI[8 * 3 * P * P];
    __shared__ double sb[4][2][NN];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int i = threadIdx.x; i < 8 * 3 * P * P; i += 256) sI[i] = interp[i];
    __syncthreads();
    const int parent = blockIdx.x * 4 + wave;
    if (parent >= np) return;  // after the workgroup's only barrier
    double* b0 = sb[wave][0];
    double* b1 = sb[wave][1];
    double acc[PER];
#pragma unroll
    for (int t = 0; t < PER; ++t) acc[t] = 0.;
    const int c0 = cstart[parent], c1 = cstart[parent + 1];
    for (int ch = c0; ch < c1; ++ch) {
        const int cidx = static_cast<int>(ckeys[ch] & 7u);
        const double* Sx = sI + (cidx * 3 + 0) * P * P;
        const double* Sy = sI + (cidx * 3 + 1) * P * P;
        const double* Sz = sI + (cidx * 3 + 2) * P * P;
        for (int i = lane; i < NN; i += 64) b0[i] = Mc[static_cast<int64_t>(ch) * LD + i];
        wave_lds_order();
        for (int idx = lane; idx < NN; idx += 64) {  // x
            const int nx = idx % P, rest = idx / P;
            double s = 0.;
#pragma unroll
            for (int m = 0; m < P; ++m) s += Sx[nx * P + m] * b0[rest * P + m];
            b1[idx] = s;
        }
        wave_lds_order();
        for (int idx = lane; idx < NN; idx += 64) {  // y
            const int i = idx % P, ny = (idx / P) % P, k = idx / (P * P);
            double s = 0.;
#pragma unroll
            for (int m = 0; m < P; ++m) s += Sy[ny * P + m] * b1[k * P * P + m * P + i];
            b0[idx] = s;
        }
        wave_lds_order();
#pragma unroll
        for (int t = 0; t < PER; ++t) {  // z
            const int idx = lane + 64 * t;
            if (idx < NN) {
                const int i = idx % P, j = (idx / P) % P, nz = idx / (P * P);
                double s = 0.;
#pragma unroll
                for (int m = 0; m < P; ++m) s += Sz[nz * P + m] * b0[m * P * P + j * P + i];
                acc[t] += s;
            }
        }
        wave_lds_order();
    }
#pragma unroll
    for (int t = 0; t < PER; ++t) {
        const int idx = lane + 64 * t;
        if (idx < LD) Mp[static_cast<int64_t>(parent) * LD + idx] = idx < NN ? acc[t] : 0.;  // zero padding
    }
}

// L2L: child[m] += sum_n Sx[nx][mx] Sy[ny][my] Sz[nz][mz] parent[n].
template <int P>
__global__ __launch_bounds__(256) void k_l2l(int np, const int32_t* __restrict__ cstart,
                                            const uint64_t* __restrict__ ckeys, const double* __restrict__ interp,
                                            const double* __restrict__ Lp, double* __restrict__ Lc, int LD) {
    constexpr int NN = P * P * P;
    __shared__ double sI[8 * 3 * P * P];
    __shared__ double sb[4][3][NN];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int i = threadIdx.x; i < 8 * 3 * P * P; i += 256) sI[i] = interp[i];
    __syncthreads();
    const int parent = blockIdx.x * 4 + wave;
    if (parent >= np) return;  // after the workgroup's only barrier
    double* par = sb[wave][0];
    double* b1 = sb[wave][1];
    double* b2 = sb[wave][2];
    for (int i = lane; i < NN; i += 64) par[i] = Lp[static_cast<int64_t>(parent) * LD + i];
    wave_lds_order();
    const int c0 = cstart[parent], c1 = cstart[parent + 1];
    for (int ch = c0; ch < c1; ++ch) {
        const int cidx = static_cast<int>(ckeys[ch] & 7u);
        const double* Sx = sI + (cidx * 3 + 0) * P * P;
        const double* Sy = sI + (cidx * 3 + 1) * P * P;
        const double* Sz = sI + (cidx * 3 + 2) * P * P;
        for (int idx = lane; idx < NN; idx += 64) {  // x
            const int mx = idx % P, rest = idx / P;
            double s = 0.;
#pragma unroll
            for (int nn = 0; nn < P; ++nn) s += Sx[nn * P + mx] * par[rest * P + nn];
            b1[idx] = s;
        }
        wave_lds_order();
        for (int idx = lane; idx < NN; idx += 64) {  // y
            const int i = idx % P, my = (idx / P) % P, k = idx / (P * P);
            double s = 0.;
#pragma unroll
            for (int nn = 0; nn < P; ++nn) s += Sy[nn * P + my] * b1[k * P * P + nn * P + i];
            b2[idx] = s;
        }
        wave_lds_order();
        for (int idx = lane; idx < NN; idx += 64) {  // z
            const int i = idx % P, j = (idx / P) % P, mz = idx / (P * P);
            double s = 0.;
#pragma unroll
            for (int nn = 0; nn < P; ++nn) s += Sz[nn * P + mz] * b2[nn * P * P + j * P + i];
            Lc[static_cast<int64_t>(ch) * LD + idx] += s;
        }
        wave_lds_order();
    }
}

// ---------------------------------------------------------------------------
// L2P: one lane per sorted particle; adds into the sorted results.
//   phi = sum_k Sz_k sum_j Sy_j sum_i Sx_i L[k][j][i], gradients with dS on one
// axis; Sx, dSx, Sy, dSy stay in registers, Sz and dSz are formed per k.
// Leaves hold from one to thousands of particles (a Plummer tree of 10M
// particles at height 8: 1.13M leaves, 641k of them with one particle), so a
// wave per leaf would leave most lanes idle.  Each lane reads its leaf's local
// expansion straight from memory: the lanes of one leaf read the same
// addresses (one fetch for the wave), the lanes of small leaves their own.
template <int P>
__global__ __launch_bounds__(256) void k_l2p(int64_t n, const int32_t* __restrict__ pleaf,
                                            const uint64_t* __restrict__ lkeys, const double* __restrict__ sp, Box bx,
                                            const double* __restrict__ Troots, const double* __restrict__ L, int LD,
                                            double* __restrict__ res) {
    __shared__ double sT[P * P];
    for (int i = threadIdx.x; i < P * P; i += 256) sT[i] = Troots[i];
    __syncthreads();
    const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (e < n) {
        const int leaf = pleaf[e];
        double a[3], b[3];
        leaf_bounds(bx, lkeys[leaf], a, b);
        const double* __restrict__ sL = L + static_cast<int64_t>(leaf) * LD;
        const double pos[3] = {sp[e], sp[n + e], sp[2 * n + e]};
        double Sx[P], dSx[P], Sy[P], dSy[P];
        const double xi0 = (2. * pos[0] - b[0] - a[0]) / (b[0] - a[0]);
        const double xi1 = (2. * pos[1] - b[1] - a[1]) / (b[1] - a[1]);
        const double xi2 = (2. * pos[2] - b[2] - a[2]) / (b[2] - a[2]);
        interp_weights<P, true>(xi0, sT, Sx, dSx);
        interp_weights<P, true>(xi1, sT, Sy, dSy);
        // T_o(xi2) and o U_{o-1}(xi2) for the z weights
        double Tz[P], dTz[P];
        {
            double t0 = 1., t1 = xi2, u0 = 1., u1 = 2. * xi2;
            Tz[0] = 1.;
            dTz[0] = 0.;
            if (P > 1) { Tz[1] = xi2; dTz[1] = 1.; }
#pragma unroll
            for (int o = 2; o < P; ++o) {
                const double t2 = 2. * xi2 * t1 - t0;
                t0 = t1; t1 = t2;
                Tz[o] = t2;
                dTz[o] = o * u1;
                const double u2 = 2. * xi2 * u1 - u0;
                u0 = u1; u1 = u2;
            }
        }
        double ph = 0., gx = 0., gy = 0., gz = 0.;
#pragma unroll 1
        for (int k = 0; k < P; ++k) {
            double sz = 1. / P, dsz = 0.;
#pragma unroll
            for (int o = 1; o < P; ++o) {
                const double t = sT[o * P + k];
                sz += 2. / P * Tz[o] * t;
                dsz += 2. / P * dTz[o] * t;
            }
            double tp = 0., tx = 0., ty = 0.;
#pragma unroll
            for (int j = 0; j < P; ++j) {
                double va = 0., vb = 0.;
#pragma unroll
                for (int i = 0; i < P; ++i) {
                    const double l = sL[(k * P + j) * P + i];
                    va += l * Sx[i];
                    vb += l * dSx[i];
                }
                tp += va * Sy[j];
                tx += vb * Sy[j];
                ty += va * dSy[j];
            }
            ph += tp * sz;
            gx += tx * sz;
            gy += ty * sz;
            gz += tp * dsz;
        }
        res[e] += ph;
        res[n + e] += gx * (2. / (b[0] - a[0]));
        res[2 * n + e] += gy * (2. / (b[1] - a[1]));
        res[3 * n + e] += gz * (2. / (b[2] - a[2]));
    }
}

// L2P on the uniform (Lagrange) basis (FUnifInterpolator.hpp:476-640,
// applyL2P + applyL2PGradient): one lane per sorted particle, the leaf's local
// expansion read directly as in k_l2p.
template <int P>
__global__ __launch_bounds__(256) void k_l2p_lagrange(int64_t n, const int32_t* __restrict__ pleaf,
                                                     const uint64_t* __restrict__ lkeys,
                                                     const double* __restrict__ sp, Box bx,
                                                     const double* __restrict__ uroots, const double* __restrict__ L,
                                                     int LD, double* __restrict__ res) {
    __shared__ double sR[P];
    if (threadIdx.x < P) sR[threadIdx.x] = uroots[threadIdx.x];
    __syncthreads();
    const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (e < n) {
        const int leaf = pleaf[e];
        double a[3], b[3];
        leaf_bounds(bx, lkeys[leaf], a, b);
        const double* __restrict__ sL = L + static_cast<int64_t>(leaf) * LD;
        const double pos[3] = {sp[e], sp[n + e], sp[2 * n + e]};
        double S[3][P], dS[3][P];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double xi = (2. * pos[d] - b[d] - a[d]) / (b[d] - a[d]);
            lagrange_weights<P, true>(xi, sR, S[d], dS[d]);
        }
        double ph = 0., gx = 0., gy = 0., gz = 0.;
        for (int k = 0; k < P; ++k)
#pragma unroll
            for (int j = 0; j < P; ++j) {
                double va = 0., vb = 0.;
#pragma unroll
                for (int i = 0; i < P; ++i) {
                    const double l = sL[(k * P + j) * P + i];
                    va += l * S[0][i];
                    vb += l * dS[0][i];
                }
                ph += va * S[1][j] * S[2][k];
                gx += vb * S[1][j] * S[2][k];
                gy += va * dS[1][j] * S[2][k];
                gz += va * S[1][j] * dS[2][k];
            }
        res[e] += ph;
        res[n + e] += gx * (2. / (b[0] - a[0]));
        res[2 * n + e] += gy * (2. / (b[1] - a[1]));
        res[3 * n + e] += gz * (2. / (b[2] - a[2]));
    }
}

// ---------------------------------------------------------------------------
// P2P of the targets in leaves of at most kP2PBig particles: kP2PLanes lanes per
// target, sources over its own leaf and the 26 neighbour slots; writes
// (initialises) the sorted results of R charge vectors, the pair geometry once
// per pair.  Leaves of at most kP2PShort particles are dealt to the lanes one by
// one (lane g: slots g - 1, g + 7, ..), the sources of longer ones are spread over
// the lanes, and the lanes' sums are added in a fixed order: the same bits for
// every n, R and device.  One lane per target walked its 27 leaves in a chain of
// dependent loads: 111 us for 1,000 particles at height 3, 520 us for 1M at height
// 7, whose pairs take 70 us to issue.
// charge(j, r): vector r's charge of sorted particle j.
constexpr int kP2PLanes = 8;
constexpr int kP2PShort = 5;

template <int R>
__device__ __forceinline__ void lane_sums(double (&v)[R], int g) {
    static_assert((R & (R - 1)) == 0, "vectors shared out by halves");
    int left = R;
#pragma unroll
    for (int d = 1; d < kP2PLanes; d <<= 1) {
        if (left > 1) {
            const bool odd = g & d;
#pragma unroll
            for (int k = 0; k < R / 2; ++k) {
                if (k >= left / 2) break;
                const double keep = odd ? v[2 * k + 1] : v[2 * k], give = odd ? v[2 * k] : v[2 * k + 1];
                v[k] = keep + __shfl_xor(give, d);
            }
            left /= 2;
        } else {
            v[0] += __shfl_xor(v[0], d);
        }
    }  // lane g: vectors g, g + kP2PLanes, ..
}

template <int R, class Charge>
__device__ __forceinline__ void p2p_f64_target(int64_t n, int64_t i, int g, const int32_t* __restrict__ pleaf,
                                               const int32_t* __restrict__ lstart, const int32_t* __restrict__ slots,
                                               const double* __restrict__ sp, Charge charge, double* __restrict__ res) {
    const int li = pleaf[i];
    if (lstart[li + 1] - lstart[li] > kP2PBig) return;  // the big leaves' kernels
    const double tx = sp[i], ty = sp[n + i], tz = sp[2 * n + i];
    double pot[R], fx[R], fy[R], fz[R];
#pragma unroll
    for (int r = 0; r < R; ++r) pot[r] = fx[r] = fy[r] = fz[r] = 0.;
    auto pair = [&](int j) {
        const double dx = tx - sp[j], dy = ty - sp[n + j], dz = tz - sp[2 * n + j];
        const double inv = rsqrt_f64_any(dx * dx + dy * dy + dz * dz);
        const double inv3 = inv * inv * inv;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const double qs = charge(j, r);
            pot[r] += inv * qs;
            fx[r] += -inv3 * dx * qs;
            fy[r] += -inv3 * dy * qs;
            fz[r] += -inv3 * dz * qs;
        }
    };
    auto leaf_of = [&](int s) { return s < 0 ? li : slots[static_cast<int64_t>(li) * kNbrSlots + s]; };
    uint32_t longer = 0;  // bit s + 1: slot s holds more than kP2PShort particles
    for (int s = g - 1; s < kNbrSlots; s += kP2PLanes) {
        const int nb = leaf_of(s);
        if (nb < 0) continue;
        const int j0 = lstart[nb], j1 = lstart[nb + 1];
        if (j1 - j0 > kP2PShort) {
            longer |= 1u << (s + 1);
            continue;
        }
        for (int j = j0; j < j1; ++j)
            if (j != i) pair(j);
    }
#pragma unroll
    for (int d = 1; d < kP2PLanes; d <<= 1) longer |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(longer), d));
    for (; longer; longer &= longer - 1) {
        const int nb = leaf_of(__ffs(longer) - 2);
        const int j1 = lstart[nb + 1];
        for (int j = lstart[nb] + g; j < j1; j += kP2PLanes)
            if (j != i) pair(j);
    }
    // The lanes' sums, over the lane bits from the lowest: while there are vectors
    // to share out, a lane keeps those with its own bit and takes the other
    // lane's sums of them, then all lanes of a vector add.  Every vector's sum is
    // the same tree over the lanes, whatever R.
    lane_sums<R>(pot, g);
    lane_sums<R>(fx, g);
    lane_sums<R>(fy, g);
    lane_sums<R>(fz, g);
    if (g >= R) return;
#pragma unroll
    for (int k = 0; k < (R > kP2PLanes ? R / kP2PLanes : 1); ++k) {
        double* o = res + static_cast<int64_t>(g + kP2PLanes * k) * 4 * n;
        o[i] = pot[k];
        o[n + i] = fx[k];
        o[2 * n + i] = fy[k];
        o[3 * n + i] = fz[k];
    }
}

__global__ __launch_bounds__(256) void k_p2p_f64(int64_t n, const int32_t* __restrict__ pleaf,
                                                const int32_t* __restrict__ lstart, const int32_t* __restrict__ slots,
                                                const double* __restrict__ sp, double* __restrict__ res) {
    const int64_t i = thread_of_grid256() / kP2PLanes;
    if (i >= n) return;
    p2p_f64_target<1>(n, i, threadIdx.x % kP2PLanes, pleaf, lstart, slots, sp, [&](int j, int) { return sp[3 * n + j]; }, res);
}

// qc: the chunk's sorted charges as [n][R]; res: the results of its first
// vector, the next vectors 4n further each.
template <int R>
__global__ __launch_bounds__(256) void k_p2p_f64_rhs(int64_t n, const int32_t* __restrict__ pleaf,
                                                    const int32_t* __restrict__ lstart,
                                                    const int32_t* __restrict__ slots, const double* __restrict__ sp,
                                                    const double* __restrict__ qc, double* __restrict__ res) {
    const int64_t i = thread_of_grid256() / kP2PLanes;
    if (i >= n) return;
    p2p_f64_target<R>(n, i, threadIdx.x % kP2PLanes, pleaf, lstart, slots, sp,
                      [&](int j, int r) { return qc[static_cast<int64_t>(j) * R + r]; }, res);
}

// P2P of the big leaves (more than kP2PBig particles).  Each wave takes work
// items of kP2PItem consecutive targets of one leaf (two per lane) and walks
// the 27 neighbour leaves in blocks of 8 sources.  Every source address is
// wave-uniform, so the sources arrive through scalar loads into SGPRs and
// feed the FP64 arithmetic as scalar operands (no LDS, no barriers).  A block
// running past the leaf's end masks the extra sources (the sorted arrays are
// padded with zeros, so the reads stay in bounds and find numbers).
constexpr int kP2PBlock64 = 8;

template <bool MASK>
__device__ __forceinline__ void pair_f64(const double (&t)[3], double sx, double sy, double sz, double sq, bool skip,
                                         double (&acc)[4]) {
    const double dx = t[0] - sx, dy = t[1] - sy, dz = t[2] - sz;
    double inv = rsqrt_f64(dx * dx + dy * dy + dz * dz);
    if (MASK) inv = skip ? 0. : inv;
    const double qi = sq * inv;
    const double qi3 = qi * inv * inv;
    acc[0] += qi;
    acc[1] -= qi3 * dx;
    acc[2] -= qi3 * dy;
    acc[3] -= qi3 * dz;
}

template <bool SELF, int T>
__device__ __forceinline__ void p2p_f64_leaf(const double* __restrict__ sp, int64_t n, int j0, int j1,
                                             const double (&t)[T][3], const int (&ti)[T], double (&acc)[T][4]) {
    int jb = j0;
    for (; jb + kP2PBlock64 <= j1; jb += kP2PBlock64) {
#pragma unroll
        for (int jj = 0; jj < kP2PBlock64; ++jj) {
            const int j = jb + jj;
            const double sx = sp[j], sy = sp[n + j], sz = sp[2 * n + j], sq = sp[3 * n + j];
#pragma unroll
            for (int u = 0; u < T; ++u) pair_f64<SELF>(t[u], sx, sy, sz, sq, j == ti[u], acc[u]);
        }
    }
    if (jb < j1) {
#pragma unroll
        for (int jj = 0; jj < kP2PBlock64; ++jj) {
            const int j = jb + jj;
            const double sx = sp[j], sy = sp[n + j], sz = sp[2 * n + j], sq = sp[3 * n + j];
            const bool past = j >= j1;
#pragma unroll
            for (int u = 0; u < T; ++u) pair_f64<true>(t[u], sx, sy, sz, sq, past || (SELF && j == ti[u]), acc[u]);
        }
    }
}

__global__ __launch_bounds__(256) void k_p2p_f64_big(const int2* __restrict__ items, const int32_t* __restrict__ nitems,
                                                    const int32_t* __restrict__ lstart,
                                                    const int32_t* __restrict__ slots, const double* __restrict__ sp,
                                                    int64_t n, double* __restrict__ res) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int total = *nitems;
    for (int it = blockIdx.x * 4 + wave; it < total; it += gridDim.x * 4) {
        const int2 item = items[it];
        const int leaf = __builtin_amdgcn_readfirstlane(item.x);
        const int first = __builtin_amdgcn_readfirstlane(item.y);
        const int tend = min(lstart[leaf + 1], first + kP2PItem);
        int ti[2];
        double t[2][3], acc[2][4];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            ti[u] = first + 64 * u + lane;
            const int tt = ti[u] < tend ? ti[u] : first;
            for (int d = 0; d < 3; ++d) t[u][d] = sp[d * n + tt];
            for (int k = 0; k < 4; ++k) acc[u][k] = 0.;
        }
        for (int s = -1; s < kNbrSlots; ++s) {
            const int nb =
                __builtin_amdgcn_readfirstlane(s < 0 ? leaf : slots[static_cast<int64_t>(leaf) * kNbrSlots + s]);
            if (nb < 0) continue;
            const int j0 = __builtin_amdgcn_readfirstlane(lstart[nb]);
            const int j1 = __builtin_amdgcn_readfirstlane(lstart[nb + 1]);
            if (s < 0)
                p2p_f64_leaf<true>(sp, n, j0, j1, t, ti, acc);
            else
                p2p_f64_leaf<false>(sp, n, j0, j1, t, ti, acc);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if (ti[u] >= tend) continue;
            res[ti[u]] = acc[u][0];
            res[n + ti[u]] = acc[u][1];
            res[2 * n + ti[u]] = acc[u][2];
            res[3 * n + ti[u]] = acc[u][3];
        }
    }
}

// Mutual FP64 P2P of the big leaves: each unordered pair of two big neighbour
// leaves once, for both particles, in the scheme of the mixed form's kernel (p2p_mixed.hip): a work item is
// up to 64 T targets of big leaf A, stationary in registers; its own leaf and
// its small neighbours are evaluated pair by pair; each big forward neighbour B
// (slots 0..12) is streamed in chunks of 64 sources, staged twice in a row in
// the wave's LDS, so that at step k lane i reads source (i + k) mod 64.  The
// source-side sum moves one lane down per step with its source, so that after
// 64 steps lane i holds the sum of source (i + 63) mod 64 and writes it to B's
// slot for this item; k_p2p_f64_combine adds a particle's slots in order: no
// atomics, the same bits on every run.  FP64 needs no phases.
// Issue slots of 4 cycles per unordered pair, T = 4: 3 differences, 3 for r^2,
// 4 for v_rsq_f64, 5 refinement, 2 for 1/r^3, 2 charge products, 8 FMAs, 3 for
// the rotation (8 DPP moves and 4 adds per source and step) = 30, against 2 x 22
// for two ordered pairs: 21.5 ms for the 2.8e10 unordered pairs of 1.25M Plummer
// particles at height 7, of which it takes 24.7 ms (the ordered kernel 56 ms).
__device__ __forceinline__ double rol1_f64(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b), 0x134, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), 0x134, 0xF, 0xF, false);
    return __builtin_bit_cast(double, (static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) | static_cast<uint32_t>(lo));
}

template <int T>
__device__ __forceinline__ void p2p_f64_mutual_item(const int32_t* __restrict__ lstart, const int32_t* __restrict__ slots,
                                                    const double* __restrict__ sp, int64_t n,
                                                    const int32_t* __restrict__ csoff,
                                                    const int64_t* __restrict__ csbase, d4* __restrict__ cpart,
                                                    double* __restrict__ res, double2* sxy, double2* szq, int leaf,
                                                    int first, int tend, int tile, int part, int parts, int lane) {
    int ti[T];
    double t[T][3], qt[T], acc[T][4];
#pragma unroll
    for (int u = 0; u < T; ++u) {
        ti[u] = first + 64 * u + lane;
        const bool ok = ti[u] < tend;  // past the item: a copy of its first target with charge 0, never written
        const int tt = ok ? ti[u] : first;
        for (int d = 0; d < 3; ++d) t[u][d] = sp[d * n + tt];
        qt[u] = ok ? sp[3 * n + tt] : 0.;
        for (int k = 0; k < 4; ++k) acc[u][k] = 0.;
    }
    const int l0 = __builtin_amdgcn_readfirstlane(lstart[leaf]), l1 = __builtin_amdgcn_readfirstlane(lstart[leaf + 1]);
    // the part's range of the chunks of 64 sources: the leaf's own, then those of
    // its big forward neighbours
    int nchunk = (l1 - l0 + 63) / 64;
    for (int s = 0; s < kNbrForward; ++s) {
        const int nb = __builtin_amdgcn_readfirstlane(slots[static_cast<int64_t>(leaf) * kNbrSlots + s]);
        if (nb < 0) continue;
        const int nbn = __builtin_amdgcn_readfirstlane(lstart[nb + 1] - lstart[nb]);
        if (nbn > kP2PBig) nchunk += (nbn + 63) / 64;
    }
    int c0 = static_cast<int>(static_cast<int64_t>(part) * nchunk / parts);
    int c1 = static_cast<int>(static_cast<int64_t>(part + 1) * nchunk / parts);
    // ordered pairs: the leaf itself, and in part 0 its small neighbours
    if (l0 + 64 * c0 < l1) p2p_f64_leaf<true, T>(sp, n, l0 + 64 * c0, min(l1, l0 + 64 * c1), t, ti, acc);
    for (int s = 0; s < (part ? 0 : kNbrSlots); ++s) {
        const int nb = __builtin_amdgcn_readfirstlane(slots[static_cast<int64_t>(leaf) * kNbrSlots + s]);
        if (nb < 0) continue;
        const int j0 = __builtin_amdgcn_readfirstlane(lstart[nb]);
        const int j1 = __builtin_amdgcn_readfirstlane(lstart[nb + 1]);
        if (j1 - j0 <= kP2PBig) p2p_f64_leaf<false, T>(sp, n, j0, j1, t, ti, acc);
    }
    c0 -= (l1 - l0 + 63) / 64;
    c1 -= (l1 - l0 + 63) / 64;
    // mutual pairs: the big forward neighbours
    for (int s = 0; s < kNbrForward && c1 > 0; ++s) {
        const int nb = __builtin_amdgcn_readfirstlane(slots[static_cast<int64_t>(leaf) * kNbrSlots + s]);
        if (nb < 0) continue;
        const int j0 = __builtin_amdgcn_readfirstlane(lstart[nb]);
        const int j1 = __builtin_amdgcn_readfirstlane(lstart[nb + 1]);
        const int nbn = j1 - j0;
        if (nbn <= kP2PBig) continue;
        const int jbeg = j0 + 64 * max(c0, 0), jend = min(j1, j0 + 64 * c1);
        c0 -= (nbn + 63) / 64;
        c1 -= (nbn + 63) / 64;
        // this item's slot in B (A is B's backward neighbour in slot 25 - s)
        const int slot = __builtin_amdgcn_readfirstlane(csoff[static_cast<int64_t>(nb) * kNbrForward + 12 - s]) + tile;
        d4* cp = cpart + (csbase[nb] + static_cast<int64_t>(slot) * nbn);
        for (int cb = jbeg; cb < jend; cb += 64) {
            const int js = cb + lane;
            const int jj = js < j1 ? js : j0;  // past the leaf: a charge-free copy of its first source
            const double2 xy = make_double2(sp[jj], sp[n + jj]);
            const double2 zq = make_double2(sp[2 * n + jj], js < j1 ? sp[3 * n + jj] : 0.);
            sxy[lane] = sxy[lane + 64] = xy;
            szq[lane] = szq[lane + 64] = zq;
            // the wave's LDS accesses run in order; the fence keeps the compiler
            // from moving other lanes' reads above these writes
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            double sa[4] = {0., 0., 0., 0.};
#pragma unroll 8
            for (int k = 0; k < 64; ++k) {
                const double2 a = sxy[lane + k], b = szq[lane + k];
                double cs[4];
#pragma unroll
                for (int u = 0; u < T; ++u) {
                    const double dx = t[u][0] - a.x, dy = t[u][1] - a.y, dz = t[u][2] - b.x;
                    const double inv = rsqrt_f64(fma(dz, dz, fma(dy, dy, dx * dx)));
                    const double inv3 = inv * (inv * inv);
                    const double a3 = b.y * inv3, b3 = qt[u] * inv3;
                    acc[u][0] = fma(b.y, inv, acc[u][0]);
                    acc[u][1] = fma(-a3, dx, acc[u][1]);
                    acc[u][2] = fma(-a3, dy, acc[u][2]);
                    acc[u][3] = fma(-a3, dz, acc[u][3]);
                    cs[0] = u ? fma(qt[u], inv, cs[0]) : qt[u] * inv;
                    cs[1] = u ? fma(b3, dx, cs[1]) : b3 * dx;
                    cs[2] = u ? fma(b3, dy, cs[2]) : b3 * dy;
                    cs[3] = u ? fma(b3, dz, cs[3]) : b3 * dz;
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) sa[q] = rol1_f64(sa[q]) + cs[q];
            }
            const int jo = cb + ((lane + 63) & 63);
            if (jo < j1) cp[jo - j0] = d4{sa[0], sa[1], sa[2], sa[3]};
            // the next chunk rewrites the sources only after these reads
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
    }
    // part 0 starts the results, the others fill the leaf's last slots
    d4* own = cpart + (csbase[leaf + 1] - static_cast<int64_t>(parts - part) * (l1 - l0) - l0);
#pragma unroll
    for (int u = 0; u < T; ++u) {
        if (ti[u] >= tend) continue;
        if (part) {
            own[ti[u]] = d4{acc[u][0], acc[u][1], acc[u][2], acc[u][3]};
            continue;
        }
        res[ti[u]] = acc[u][0];
        res[n + ti[u]] = acc[u][1];
        res[2 * n + ti[u]] = acc[u][2];
        res[3 * n + ti[u]] = acc[u][3];
    }
}

__global__ __launch_bounds__(256) void k_p2p_f64_mutual(const int2* __restrict__ items, const int32_t* __restrict__ claims,
                                                       int total, const int32_t* __restrict__ lstart,
                                                       const int32_t* __restrict__ slots, const double* __restrict__ sp,
                                                       int64_t n, const int32_t* __restrict__ csoff,
                                                       const int64_t* __restrict__ csbase,
                                                       const int32_t* __restrict__ csparts, d4* __restrict__ cpart,
                                                       int32_t* __restrict__ next, double* __restrict__ res) {
    static_assert(kP2PMutualItem == 256, "work item = one wave x up to 4 targets");
    __shared__ double2 s_xy[4][128], s_zq[4][128];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // parts of work items claimed one at a time, costliest items first; every wave
    // leaves once the counter passes the last
    for (;;) {
        int at = 0;
        if (lane == 0) at = atomicAdd(next, 1);
        at = __builtin_amdgcn_readfirstlane(at);
        if (at >= total) break;
        const int claim = __builtin_amdgcn_readfirstlane(claims[at]);
        const int part = claim % kP2PMaxParts;
        const int2 item = items[claim / kP2PMaxParts];
        const int leaf = __builtin_amdgcn_readfirstlane(item.x);
        const int first = __builtin_amdgcn_readfirstlane(item.y);
        const int parts = __builtin_amdgcn_readfirstlane(csparts[leaf]);
        const int l0 = __builtin_amdgcn_readfirstlane(lstart[leaf]);
        const int tend = min(__builtin_amdgcn_readfirstlane(lstart[leaf + 1]), first + kP2PMutualItem);
        const int tile = (first - l0) / kP2PMutualItem;
        // as many targets per lane as the item needs: the last item of a leaf
        // may hold a few
#define ITEM(T) \
    p2p_f64_mutual_item<T>(lstart, slots, sp, n, csoff, csbase, cpart, res, s_xy[wave], s_zq[wave], leaf, first, tend, tile, part, \
                           parts, lane)
        switch ((tend - first + 63) / 64) {
            case 1: ITEM(1); break;
            case 2: ITEM(2); break;
            case 3: ITEM(3); break;
            default: ITEM(4); break;
        }
#undef ITEM
    }
}

// Adds the source-side sums of the mutual P2P to the big leaves' particles: one
// thread per particle, its slots in order.
__global__ __launch_bounds__(256) void k_p2p_f64_combine(int64_t n, const int32_t* __restrict__ pleaf,
                                                        const int32_t* __restrict__ lstart,
                                                        const int64_t* __restrict__ csbase,
                                                        const d4* __restrict__ cpart, double* __restrict__ res) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int li = pleaf[i];
    const int j0 = lstart[li], m = lstart[li + 1] - j0;
    if (m <= kP2PBig) return;
    const int64_t b0 = csbase[li];
    const int64_t ns = (csbase[li + 1] - b0) / m;
    if (ns == 0) return;
    const d4* p = cpart + b0 + (i - j0);
    d4 s = {0., 0., 0., 0.};
    for (int64_t k = 0; k < ns; ++k) s += p[k * m];
    for (int q = 0; q < 4; ++q) res[q * n + i] += s[q];
}

__global__ void k_mfma_probe(double* out) {
    const int l = threadIdx.x;
    const double a = 1.0 + (l % 16) * 4 + (l / 16);    // A[l%16][l/16]
    const double b = 0.5 + (l / 16) * 16 + (l % 16);    // B[l/16][l%16]
    d4 c = {0., 0., 0., 0.};
    c = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    for (int i = 0; i < 4; ++i) out[(4 * i + l / 16) * 16 + (l % 16)] = c[i];
}

// Sorted -> input order.  The passes accumulate the potential and the field
// grad(phi); the force is q grad(phi) (the reference's convention,
// FP2P.hpp:80-101: F_t += q_t q_s grad_t(1/r)), the field is kept as well.
// One thread per input index o reads its sorted index i = iperm[o]: the seven
// outputs are written contiguously and the five inputs gathered.
__global__ __launch_bounds__(256) void k_scatter(int64_t n, const int32_t* __restrict__ iperm,
                                                const double* __restrict__ sp, const double* __restrict__ rs,
                                                double* __restrict__ r, double* __restrict__ field) {
    const int64_t o = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (o >= n) return;
    const int64_t i = iperm[o];
    const double q = sp[3 * n + i];
    r[o] = rs[i];
    for (int d = 1; d < 4; ++d) {
        const double g = rs[d * n + i];
        r[d * n + o] = g * q;
        field[(d - 1) * n + o] = g;
    }
}

inline unsigned blocks256(int64_t n) { return static_cast<unsigned>((n + 255) / 256); }

// Grid-stride fill with zeros (a kernel node, where hipMemsetAsync would be a
// memset node in a captured graph).
__global__ __launch_bounds__(256) void k_zero_words(uint32_t* __restrict__ p, int64_t words) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < words; i += stride) p[i] = 0u;
}

// Grid-stride copy (ADD = false) or sum (ADD = true) of count doubles.
template <bool ADD>
__global__ __launch_bounds__(256) void k_combine(double* __restrict__ dst, const double* __restrict__ src,
                                                 int64_t count) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += stride)
        dst[i] = ADD ? dst[i] + src[i] : src[i];
}

}  // namespace

Box make_box(const Context* c) {
    Box b;
    const double half = c->P.box_width / 2;
    for (int d = 0; d < 3; ++d) b.corner[d] = c->P.box_center[d] + (-half);
    const int Lloc = c->P.tree_height - 1;
    b.leafw = c->P.box_width / static_cast<double>(1 << Lloc);
    b.cmask = (1u << Lloc) - 1u;
    return b;
}

M2LLevels make_levels(const Context* c, int tile_targets, int& tiles) {
    const int L = c->height() - 1;
    M2LLevels lv{};
    lv.nlev = 0;
    tiles = 0;
    lv.tile_begin[0] = 0;
    // the M2L levels of the working range (every level top..h-1 by default)
    const int lo = c->work_upper > c->top() ? c->work_upper : c->top();
    const int hi = c->work_lower > 0 && c->work_lower - 1 < L ? c->work_lower - 1 : L;
    for (int l = lo; l <= hi; ++l) {
        const int i = lv.nlev++;
        lv.cell_off[i] = c->lvl_off[l];
        lv.pcount_off[i] = 8 * l;
        // 2^l cells per axis of a set: scale factor 2 / (width / 2^l) (FInterpMatrixKernel.hpp:124-133)
        const int lloc = l - c->set_levels;
        lv.scale[i] = 2. / (c->P.box_width / static_cast<double>(int64_t(1) << lloc));
        // segment of 8 x (tiles of the largest parity); the parity counts are
        // on the device, ceil(ncell/tile) bounds every parity's tile count
        tiles += 8 * static_cast<int>((c->ncell[l] + tile_targets - 1) / tile_targets);
        lv.tile_begin[i + 1] = tiles;
    }
    return lv;
}

namespace {

template <int P>
int p2m_impl(Context* c) {
    const int L = c->height() - 1;
    const int64_t nl = c->ncell[L];
    prof_begin(c, "p2m");
    auto kern = k_p2m<P, 0>;
    if constexpr (P <= kUniformMaxOrder)
        if (c->basis == 1) kern = k_p2m<P, 1>;
    (void)nl;
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>((c->n + 63) / 64)), dim3(64), 0, c->stream, c->n,
                       c->d_pleaf.as<int32_t>(), c->d_cellkey.as<uint64_t>() + c->lvl_off[L],
                       c->d_leafstart.as<int32_t>(), c->d_sorted.as<double>(), make_box(c), c->d_Troots.as<double>(),
                       c->d_uroots.as<double>(), c->d_M.as<double>() + static_cast<size_t>(c->lvl_off[L]) * c->LD,
                       c->LD);
    prof_end(c);
    return check_launch(c, "p2m");
}

template <int P>
int m2m_impl(Context* c, int l) {
    const int64_t np = c->ncell[l];
    if (np == 0) return HFMM_OK;
    prof_begin(c, "m2m");
    hipLaunchKernelGGL(k_m2m<P>, dim3(static_cast<unsigned>((np + 3) / 4)), dim3(256), 0, c->stream,
                       static_cast<int>(np), c->d_childstart.as<int32_t>() + c->cs_off[l],
                       c->d_cellkey.as<uint64_t>() + c->lvl_off[l + 1],
                       c->d_child.as<double>(), c->d_M.as<double>() + static_cast<size_t>(c->lvl_off[l + 1]) * c->LD,
                       c->d_M.as<double>() + static_cast<size_t>(c->lvl_off[l]) * c->LD, c->LD);
    prof_end(c);
    return check_launch(c, "m2m");
}

template <int P>
int l2l_impl(Context* c, int l) {
    const int64_t np = c->ncell[l];
    if (np == 0) return HFMM_OK;
    prof_begin(c, "l2l");
    hipLaunchKernelGGL(k_l2l<P>, dim3(static_cast<unsigned>((np + 3) / 4)), dim3(256), 0, c->stream,
                       static_cast<int>(np), c->d_childstart.as<int32_t>() + c->cs_off[l],
                       c->d_cellkey.as<uint64_t>() + c->lvl_off[l + 1],
                       c->d_child.as<double>(), c->d_L.as<double>() + static_cast<size_t>(c->lvl_off[l]) * c->LD,
                       c->d_L.as<double>() + static_cast<size_t>(c->lvl_off[l + 1]) * c->LD, c->LD);
    prof_end(c);
    return check_launch(c, "l2l");
}

template <int P>
int l2p_impl(Context* c) {
    const int L = c->height() - 1;
    prof_begin(c, "l2p");
    if constexpr (P <= kUniformMaxOrder) {
        if (c->basis == 1) {
            hipLaunchKernelGGL(k_l2p_lagrange<P>, dim3(blocks256(c->n)), dim3(256), 0, c->stream, c->n,
                               c->d_pleaf.as<int32_t>(), c->d_cellkey.as<uint64_t>() + c->lvl_off[L],
                               c->d_sorted.as<double>(), make_box(c), c->d_uroots.as<double>(),
                               c->d_L.as<double>() + static_cast<size_t>(c->lvl_off[L]) * c->LD, c->LD,
                               sorted_results(c));
            prof_end(c);
            return check_launch(c, "l2p");
        }
    }
    hipLaunchKernelGGL(k_l2p<P>, dim3(blocks256(c->n)), dim3(256), 0, c->stream, c->n, c->d_pleaf.as<int32_t>(),
                       c->d_cellkey.as<uint64_t>() + c->lvl_off[L], c->d_sorted.as<double>(), make_box(c),
                       c->d_Troots.as<double>(), c->d_L.as<double>() + static_cast<size_t>(c->lvl_off[L]) * c->LD,
                       c->LD, sorted_results(c));
    prof_end(c);
    return check_launch(c, "l2p");
}

#define HFMM_DISPATCH(P_, CALL)                                                   \
    switch (P_) {                                                                 \
        case 5: return CALL(5);                                                   \
        case 6: return CALL(6);                                                   \
        case 7: return CALL(7);                                                   \
        case 8: return CALL(8);                                                   \
        default: return fail(c, HFMM_ERR_ARG, "order not compiled (5..8)");      \
    }

}  // namespace

int run_p2m(Context* c) {
#define CALL(P) p2m_impl<P>(c)
    HFMM_DISPATCH(c->order(), CALL)
#undef CALL
}
int run_m2m(Context* c, int l) {
#define CALL(P) m2m_impl<P>(c, l)
    HFMM_DISPATCH(c->order(), CALL)
#undef CALL
}
int run_l2l(Context* c, int l) {
#define CALL(P) l2l_impl<P>(c, l)
    HFMM_DISPATCH(c->order(), CALL)
#undef CALL
}
int run_l2p(Context* c) {
#define CALL(P) l2p_impl<P>(c)
    HFMM_DISPATCH(c->order(), CALL)
#undef CALL
}
int run_p2p(Context* c) {
    if (!c->p2p_small_done) {
        prof_begin(c, "p2p");
        hipLaunchKernelGGL(k_p2p_f64, grid256(c->n * kP2PLanes), dim3(256), 0, c->stream, c->n, c->d_pleaf.as<int32_t>(),
                           c->d_leafstart.as<int32_t>(), c->d_p2p.as<int32_t>(), c->d_sorted.as<double>(),
                           sorted_results(c));
        prof_end(c);
        HFMM_TRY(check_launch(c, "p2p"));
    }
    if (c->p2p_items_cap == 0) return HFMM_OK;
    if (c->p2p_mutual && c->p2p_mutual_on) {
        // persistent grid: as many workgroups as fit on the device at once
        static int resident[64] = {0};
        if (c->device < 0 || c->device >= 64) return fail(c, HFMM_ERR_ARG, "device ordinal above 63");
        if (resident[c->device] == 0) {
            int per_cu = 0, cus = 0;
            HFMM_HIP(c, hipOccupancyMaxActiveBlocksPerMultiprocessor(
                            &per_cu, reinterpret_cast<const void*>(&k_p2p_f64_mutual), 256, 0));
            HFMM_HIP(c, hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device));
            resident[c->device] = std::max(1, per_cu) * std::max(1, cus);
        }
        const int64_t want = (c->p2p_claims + 3) / 4;
        const unsigned grid = static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>(want, resident[c->device])));
        HFMM_TRY(zero_device(c, p2p_mutual_next(c), sizeof(int32_t)));  // a fill kernel: capturable
        prof_begin(c, "p2p_big");
        hipLaunchKernelGGL(k_p2p_f64_mutual, dim3(grid), dim3(256), 0, c->stream, c->d_p2pitems_m.as<int2>(),
                           c->d_claims.as<int32_t>(), c->p2p_claims, c->d_leafstart.as<int32_t>(), c->d_p2p.as<int32_t>(),
                           c->d_sorted.as<double>(), c->n, c->d_csoff.as<int32_t>(), c->d_csbase.as<int64_t>(),
                           c->d_csparts.as<int32_t>(), c->d_cpart.as<d4>(), p2p_mutual_next(c), sorted_results(c));
        prof_end(c);
        HFMM_TRY(check_launch(c, "p2p_big"));
        prof_begin(c, "p2p_combine");
        hipLaunchKernelGGL(k_p2p_f64_combine, dim3(blocks256(c->n)), dim3(256), 0, c->stream, c->n,
                           c->d_pleaf.as<int32_t>(), c->d_leafstart.as<int32_t>(), c->d_csbase.as<int64_t>(),
                           c->d_cpart.as<d4>(), sorted_results(c));
        prof_end(c);
        return check_launch(c, "p2p_combine");
    }
    prof_begin(c, "p2p_big");
    hipLaunchKernelGGL(k_p2p_f64_big, dim3((p2p_tiled_grid(c) + 3) / 4), dim3(256), 0, c->stream,
                       c->d_p2pitems.as<int2>(), p2p_item_count(c), c->d_leafstart.as<int32_t>(),
                       c->d_p2p.as<int32_t>(), c->d_sorted.as<double>(), c->n, sorted_results(c));
    prof_end(c);
    return check_launch(c, "p2p_big");
}

int zero_device(Context* c, void* ptr, size_t bytes) {
    if (bytes % 4) return fail(c, HFMM_ERR_ARG, "zero_device: size not a multiple of 4");
    const int64_t words = static_cast<int64_t>(bytes / 4);
    if (words == 0) return HFMM_OK;
    const int64_t blocks = std::min<int64_t>((words + 1023) / 1024, 65536);
    hipLaunchKernelGGL(k_zero_words, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, c->stream,
                       static_cast<uint32_t*>(ptr), words);
    return check_launch(c, "zero");
}

int combine_device(Context* c, double* dst, const double* src, int64_t count, bool add) {
    if (count <= 0) return HFMM_OK;
    const int64_t blocks = std::min<int64_t>((count + 1023) / 1024, 65536);
    if (add)
        hipLaunchKernelGGL(k_combine<true>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, c->stream, dst, src,
                           count);
    else
        hipLaunchKernelGGL(k_combine<false>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, c->stream, dst, src,
                           count);
    return check_launch(c, "combine");
}

int run_p2p_small_all(Context* c) {
    HFMM_TRY(gather_all_charges(c, false));
    RhsChunk ch[HFMM_MAX_RHS];
    const int nch = rhs_chunks(c->nrhs, ch);
    const int64_t npad = (c->n + 7) & ~int64_t(7);
    prof_begin(c, "p2p_rhs");
    for (int k = 0; k < nch; ++k) {
        const double* qc = c->d_qall.as<double>() + npad * ch[k].r0;
        double* res = c->d_res_sorted.as<double>() + static_cast<size_t>(ch[k].r0) * 4 * c->n;
        const dim3 grid = grid256(c->n * kP2PLanes), block(256);
        const int32_t* pl = c->d_pleaf.as<int32_t>();
        const int32_t* ls = c->d_leafstart.as<int32_t>();
        const int32_t* sl = c->d_p2p.as<int32_t>();
        const double* sp = c->d_sorted.as<double>();
        switch (ch[k].R) {
            case 8: hipLaunchKernelGGL(k_p2p_f64_rhs<8>, grid, block, 0, c->stream, c->n, pl, ls, sl, sp, qc, res); break;
            case 4: hipLaunchKernelGGL(k_p2p_f64_rhs<4>, grid, block, 0, c->stream, c->n, pl, ls, sl, sp, qc, res); break;
            case 2: hipLaunchKernelGGL(k_p2p_f64_rhs<2>, grid, block, 0, c->stream, c->n, pl, ls, sl, sp, qc, res); break;
            default: hipLaunchKernelGGL(k_p2p_f64_rhs<1>, grid, block, 0, c->stream, c->n, pl, ls, sl, sp, qc, res); break;
        }
    }
    prof_end(c);
    return check_launch(c, "p2p_rhs");
}

int zero_results(Context* c) { return zero_device(c, sorted_results(c), sizeof(double) * 4 * c->n); }

int scatter_results(Context* c, int rhs) {
    prof_begin(c, "scatter");
    hipLaunchKernelGGL(k_scatter, dim3(blocks256(c->n)), dim3(256), 0, c->stream, c->n, c->d_iperm.as<int32_t>(),
                       c->d_sorted.as<double>(), sorted_results(c),
                       c->d_res.as<double>() + static_cast<size_t>(rhs) * 4 * c->n,
                       c->d_field.as<double>() + static_cast<size_t>(rhs) * 3 * c->n);
    prof_end(c);
    return check_launch(c, "scatter");
}

int selftest_mfma_f64(Context* c, double* out) {
    DevBuf b;
    HFMM_TRY(ensure(c, b, sizeof(double) * 256));
    hipLaunchKernelGGL(k_mfma_probe, dim3(1), dim3(64), 0, c->stream, b.as<double>());
    int st = check_launch(c, "mfma_probe");
    if (st == HFMM_OK) {
        if (hipMemcpyAsync(out, b.ptr, sizeof(double) * 256, hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
            hipStreamSynchronize(c->stream) != hipSuccess)
            st = fail(c, HFMM_ERR_DEVICE, "probe copy failed");
    }
    release(b);
    return st;
}

}  // namespace hfmm

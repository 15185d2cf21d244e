// fmm_global.hip -- the passes of the reference's FChebKernel that differ from
// the symmetric kernel's (Src/Kernels/Chebyshev/FChebKernel.hpp:93-200), FP64:
//   compression    M~ = B^T M after P2M and after each M2M      (applyB, overwrite)
//   M2L            L~ += 2/w C_t M~_src over the interaction list (applyC)
//   decompression  L += U L~ before each L2L and before L2P      (applyU, add)
// The compressed expansions have k entries per cell (the global rank).  One
// 64-lane wave per cell; lane r owns rank rows r, r + 64, ... (R of them).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "fmm_common.hpp"

namespace hfmm {
namespace {

constexpr int kMaxRankRows = 8;  // ranks up to 512 (the dense scheme's p^3 at order 8)

// M~[cell][a] = sum_n B[n][a] M[cell][n]; Bt is B as [nn][k].
template <int R>
__global__ __launch_bounds__(64) void k_global_compress(int64_t ncell, const double* __restrict__ M, int LD,
                                                        const double* __restrict__ Bt, int nn, int k,
                                                        double* __restrict__ Mt) {
    const int64_t cell = blockIdx.x;
    if (cell >= ncell) return;
    const int lane = threadIdx.x;
    double acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.;
    const double* m = M + cell * LD;
    for (int n = 0; n < nn; ++n) {
        const double v = m[n];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int a = lane + 64 * r;
            if (a < k) acc[r] += Bt[static_cast<int64_t>(n) * k + a] * v;
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int a = lane + 64 * r;
        if (a < k) Mt[cell * k + a] = acc[r];
    }
}

// L[cell][n] += sum_a U[a][n] L~[cell][a]; U as [k][nn].
__global__ __launch_bounds__(64) void k_global_decompress(int64_t ncell, const double* __restrict__ Lt, int k,
                                                          const double* __restrict__ U, int nn,
                                                          double* __restrict__ L, int LD) {
    const int64_t cell = blockIdx.x;
    if (cell >= ncell) return;
    const double* lt = Lt + cell * k;
    for (int n = threadIdx.x; n < nn; n += 64) {
        double s = 0.;
        for (int a = 0; a < k; ++a) s += U[static_cast<int64_t>(a) * nn + n] * lt[a];
        L[cell * LD + n] += s;
    }
}

// L~[cell] += scale C_pos M~[src] for every source of the cell's 189 slots, in
// slot order; slot s of a cell of parity e sits at relative position
// slotpos[e][s].  C_pos is column-major k x k.
template <int R>
__global__ __launch_bounds__(64) void k_global_m2l(int64_t ncell, const int32_t* __restrict__ slots,
                                                   const uint64_t* __restrict__ keys,
                                                   const int16_t* __restrict__ slotpos,
                                                   const double* __restrict__ C, const double* __restrict__ Mt,
                                                   int k, double scale, double* __restrict__ Lt) {
    const int64_t cell = blockIdx.x;
    if (cell >= ncell) return;
    const int lane = threadIdx.x;
    const int par = static_cast<int>(keys[cell] & 7u);
    double acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.;
    for (int s = 0; s < kFarSlots; ++s) {
        const int src = slots[cell * kFarSlots + s];
        if (src < 0) continue;  // the same for every lane
        const double* Cp = C + static_cast<int64_t>(slotpos[par * kFarSlots + s]) * k * k;
        const double* m = Mt + static_cast<int64_t>(src) * k;
        double t[R];
#pragma unroll
        for (int r = 0; r < R; ++r) t[r] = 0.;
        for (int j = 0; j < k; ++j) {
            const double mj = m[j];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int i = lane + 64 * r;
                if (i < k) t[r] += Cp[static_cast<int64_t>(j) * k + i] * mj;
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] += scale * t[r];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = lane + 64 * r;
        if (i < k) Lt[cell * k + i] += acc[r];
    }
}

// ---------------------------------------------------------------------------
// The same M2L on FP64 MFMA (v_mfma_f64_16x16x4f64), for ranks up to
// 16 kGlobalMfmaMaxTiles.  The operators are used as a padded row-major copy
// Cr[pos][i][j] (KP = 16 NR rows and columns, zeros outside k x k).  A
// workgroup of four waves owns one column tile of 16 targets of one parity at
// one level (the parity-sorted cell order of the symmetric kernel, one parity
// per XCD); wave w takes the tile's slots w, w + 4, ... and keeps all NR row
// tiles of its partial L~ in registers; the four partial sums are added in
// wave order through LDS (the same bits on every run) and added, scaled, to
// L~.  Per slot and 16-wide K block, lane (i, g) = (lane % 16, lane / 16)
// reads four consecutive entries 16 kb + 4 g + s (s < 4) of its target's M~
// (B operand) and of row i of every row tile of C (A operand): a permutation
// of the K order shared by both, so row-major loads of 32 bytes.  Register r
// of lane (i, g) holds D[4 r + g][i] (the FP64 layout the symmetric kernel's
// hfmm_selftest_mfma_f64 checks).
constexpr int kGlobalMfmaMaxTiles = 16;

typedef double d4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void k_global_pad_ops(const double* __restrict__ C, int k, int KP,
                                                        double* __restrict__ Cr) {
    const int64_t pos = blockIdx.x;
    const double* src = C + pos * k * k;
    double* dst = Cr + pos * KP * KP;
    for (int e = threadIdx.x; e < KP * KP; e += blockDim.x) {
        const int i = e / KP, j = e % KP;
        dst[e] = (i < k && j < k) ? src[static_cast<int64_t>(j) * k + i] : 0.;
    }
}

template <int NR>
__global__ __launch_bounds__(256) void k_global_m2l_mfma(M2LLevels lv, const int32_t* __restrict__ slots,
                                                        const int32_t* __restrict__ order,
                                                        const int32_t* __restrict__ pcount,
                                                        const int16_t* __restrict__ slotpos,
                                                        const double* __restrict__ Cr, const double* __restrict__ Mt,
                                                        int k, double* __restrict__ Lt) {
    constexpr int KP = 16 * NR;
    constexpr int W = 4;
    __shared__ double red[16 * KP];  // [target column][row]
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, g = lane >> 4;
    const int bid = blockIdx.x;
    if (bid >= lv.tile_begin[lv.nlev]) return;
    int li = 0;
    while (bid >= lv.tile_begin[li + 1]) ++li;
    const int lb = bid - lv.tile_begin[li];
    const int e = lb % 8;  // parity: consecutive workgroups land on different XCDs
    const int ptile = lb / 8;
    const int32_t* pc = pcount + lv.pcount_off[li];
    int first = 0;
    for (int q = 0; q < e; ++q) first += pc[q];
    const int cnt = min(16, pc[e] - ptile * 16);
    if (cnt <= 0) return;  // the same for the whole workgroup
    first += ptile * 16;
    const int64_t coff = lv.cell_off[li];
    const int32_t* lslots = slots + coff * kFarSlots;
    const double* Ml = Mt + coff * k;
    const int tgt = col < cnt ? order[coff + first + col] : -1;
    d4 acc[NR];
#pragma unroll
    for (int rt = 0; rt < NR; ++rt) acc[rt] = d4{0., 0., 0., 0.};
    for (int s = wave; s < kFarSlots; s += W) {
        const int src = tgt >= 0 ? lslots[static_cast<int64_t>(tgt) * kFarSlots + s] : -1;
        if (__ballot(src >= 0) == 0) continue;  // uniform over the wave
        const double* C = Cr + static_cast<int64_t>(slotpos[e * kFarSlots + s]) * KP * KP + col * KP + 4 * g;
        const double* m = Ml + static_cast<int64_t>(src >= 0 ? src : 0) * k;
#pragma unroll 2
        for (int kb = 0; kb < NR; ++kb) {
            double b[4];
#pragma unroll
            for (int s2 = 0; s2 < 4; ++s2) {
                const int j = 16 * kb + 4 * g + s2;
                b[s2] = (src >= 0 && j < k) ? m[j] : 0.;
            }
#pragma unroll
            for (int rt = 0; rt < NR; ++rt) {
                const d4 a = *reinterpret_cast<const d4*>(C + 16 * rt * KP + 16 * kb);
#pragma unroll
                for (int s2 = 0; s2 < 4; ++s2) acc[rt] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s2], b[s2], acc[rt], 0, 0, 0);
            }
        }
    }
    // partial sums in wave order: wave 0 writes, waves 1..3 add
    for (int w = 0; w < W; ++w) {
        if (wave == w) {
#pragma unroll
            for (int rt = 0; rt < NR; ++rt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int idx = col * KP + 16 * rt + 4 * r + g;
                    red[idx] = (w == 0 ? 0. : red[idx]) + acc[rt][r];
                }
        }
        __syncthreads();
    }
    const double scale = lv.scale[li];
    double* Ll = Lt + coff * k;
    for (int idx = tid; idx < 16 * KP; idx += 64 * W) {
        const int cc = idx / KP, i = idx % KP;
        if (cc < cnt && i < k) Ll[static_cast<int64_t>(order[coff + first + cc]) * k + i] += scale * red[idx];
    }
}

// ---------------------------------------------------------------------------
// The uniform scheme (FUnifKernel): expansions in Fourier space.  A cell's p^3
// node values, zero-padded to N^3 (N = 2p-1), are 3D-DFT'd; real input, so
// only kx < p is kept: NF = p N^2 complex entries, index kx + p (ky + N kz).
// One 64-lane wave per cell, the three axes one after the other through LDS.
// tw[j] = (cos 2 pi j/N, sin 2 pi j/N).

// M^ = DFT(pad(M)) (FUnifM2LHandler::applyZeroPaddingAndDFT), overwrite.
template <int P>
__global__ __launch_bounds__(64) void k_unif_forward(int64_t ncell, const double* __restrict__ M, int LD,
                                                     const double2* __restrict__ tw, double2* __restrict__ Mh) {
    constexpr int N = 2 * P - 1, NN = P * P * P, NF = P * N * N;
    __shared__ double sM[NN];
    __shared__ double2 sA[NN];         // [kx][b][c]: kx + P (b + P c)
    __shared__ double2 sB[P * N * P];  // [kx][ky][c]: kx + P (ky + N c)
    __shared__ double2 sW[N];
    const int64_t cell = blockIdx.x;
    if (cell >= ncell) return;
    const int lane = threadIdx.x;
    if (lane < N) sW[lane] = tw[lane];
    for (int i = lane; i < NN; i += 64) sM[i] = M[cell * LD + i];
    __syncthreads();
    for (int i = lane; i < NN; i += 64) {  // x: real -> complex
        const int kx = i % P, bc = i / P;
        double re = 0., im = 0.;
#pragma unroll
        for (int a = 0; a < P; ++a) {
            const double m = sM[a + P * bc];
            const double2 w = sW[(a * kx) % N];
            re += m * w.x;
            im -= m * w.y;
        }
        sA[i] = make_double2(re, im);
    }
    __syncthreads();
    for (int i = lane; i < P * N * P; i += 64) {  // y
        const int kx = i % P, ky = (i / P) % N, cc = i / (P * N);
        double re = 0., im = 0.;
#pragma unroll
        for (int b = 0; b < P; ++b) {
            const double2 v = sA[kx + P * (b + P * cc)];
            const double2 w = sW[(b * ky) % N];
            re += v.x * w.x + v.y * w.y;
            im += v.y * w.x - v.x * w.y;
        }
        sB[i] = make_double2(re, im);
    }
    __syncthreads();
    for (int i = lane; i < NF; i += 64) {  // z
        const int kxy = i % (P * N), kz = i / (P * N);
        double re = 0., im = 0.;
#pragma unroll
        for (int cc = 0; cc < P; ++cc) {
            const double2 v = sB[kxy + P * N * cc];
            const double2 w = sW[(cc * kz) % N];
            re += v.x * w.x + v.y * w.y;
            im += v.y * w.x - v.x * w.y;
        }
        Mh[cell * NF + i] = make_double2(re, im);
    }
}

// L += IDFT(L^) restricted to the p^3 nodes, over N^3
// (FUnifM2LHandler::unapplyZeroPaddingAndDFT + FBlas::add).
template <int P>
__global__ __launch_bounds__(64) void k_unif_inverse(int64_t ncell, const double2* __restrict__ Lh,
                                                     const double2* __restrict__ tw, double* __restrict__ L, int LD) {
    constexpr int N = 2 * P - 1, NN = P * P * P, NF = P * N * N;
    __shared__ double2 sF[NF];
    __shared__ double2 sH[P * N * P];  // [kx][ky][c]
    __shared__ double2 sG[NN];         // [kx][b][c]
    __shared__ double2 sW[N];
    const int64_t cell = blockIdx.x;
    if (cell >= ncell) return;
    const int lane = threadIdx.x;
    if (lane < N) sW[lane] = tw[lane];
    for (int i = lane; i < NF; i += 64) sF[i] = Lh[cell * NF + i];
    __syncthreads();
    for (int i = lane; i < P * N * P; i += 64) {  // z, outputs c < p
        const int kxy = i % (P * N), cc = i / (P * N);
        double re = 0., im = 0.;
#pragma unroll
        for (int kz = 0; kz < N; ++kz) {
            const double2 v = sF[kxy + P * N * kz];
            const double2 w = sW[(cc * kz) % N];
            re += v.x * w.x - v.y * w.y;
            im += v.x * w.y + v.y * w.x;
        }
        sH[i] = make_double2(re, im);
    }
    __syncthreads();
    for (int i = lane; i < NN; i += 64) {  // y, outputs b < p
        const int kx = i % P, b = (i / P) % P, cc = i / (P * P);
        double re = 0., im = 0.;
#pragma unroll
        for (int ky = 0; ky < N; ++ky) {
            const double2 v = sH[kx + P * (ky + N * cc)];
            const double2 w = sW[(b * ky) % N];
            re += v.x * w.x - v.y * w.y;
            im += v.x * w.y + v.y * w.x;
        }
        sG[i] = make_double2(re, im);
    }
    __syncthreads();
    constexpr double inv = 1. / (static_cast<double>(N) * N * N);
    for (int i = lane; i < NN; i += 64) {  // x: the Hermitian half back to real
        const int a = i % P, bc = i / P;
        double v = sG[P * bc].x;
        double h = 0.;
#pragma unroll
        for (int kx = 1; kx < P; ++kx) {
            const double2 g = sG[kx + P * bc];
            const double2 w = sW[(a * kx) % N];
            h += g.x * w.x - g.y * w.y;
        }
        v += 2. * h;
        L[cell * LD + i] += v * inv;
    }
}

// The M2L levels of one uniform-scheme launch: level i owns workgroups
// first[i] .. first[i + 1] - 1, kUnifCells target cells each.
struct UnifLevels {
    int nlev;
    int64_t first[kMaxLevels + 1];
    int ncell[kMaxLevels];
    const int32_t* slots[kMaxLevels];
    const uint64_t* keys[kMaxLevels];
    const double2* Mh[kMaxLevels];
    double2* Lh[kMaxLevels];
    double scale[kMaxLevels];
};
constexpr int kUnifCells = 32;

// L^ += scale K^_pos . M^[src] entrywise (FUnifM2LHandler::applyFC), the levels of
// many children per parent in one launch (FULL), those of few in another.  A wave takes
// the siblings of one parent (up to 8 targets) and 64 spectrum entries: for each
// of the 26 neighbour parents FULL reads the 8 source spectra once for all
// targets, and each of the 27 kernel spectra of that direction (offset 2 d + b - a
// of source child b from target child a, at most 3 values per axis) once for the 1
// to 8 pairs that have it.  One target at a time, every pair reads both: 3,024 spectra for the 8 targets
// of a full parent against 910 here, and the caches were the bound (15.7 TB/s,
// 2.13 ms at 20,000 particles, height 5, order 7; 0.56 ms now).
// A workgroup's four waves take the parents that begin in its kUnifCells cells,
// so they read the same kernel spectra at about the same time.
// Where parents have few children most of the 27 kernel spectra serve no pair: not
// FULL reads a source's spectrum once, and a kernel spectrum for each target that
// has it, which needs fewer registers too (5 waves per SIMD).  From kUnifFull
// children per parent FULL is faster, M2L in us, few / full, uniform particles at
// order 7: 1.1 children (5,000, h7) 1,141 / 2,468; 2.7 (100,000, h7) 14,804 / 23,991;
// 4.2 (192,000, h7) 21,390 / 28,248; 5.5 (38,400, h6) 3,997 / 3,776; 8 (20,000, h5)
// 815 / 582; a sphere of 30,000 at h8 2,418 / 5,260 (one target at a time 3,597).
constexpr int64_t kUnifFull = 5;

template <int P, bool FULL>
__global__ __launch_bounds__(256) void k_unif_m2l(UnifLevels lv, const int16_t* __restrict__ slotpos,
                                                  const double2* __restrict__ K) {
    constexpr int N = 2 * P - 1, NF = P * N * N;
    constexpr int kDirs = 27;
    __shared__ int s_src[4][8 * kDirs];  // source cell of (direction, child), -1: none
    const int64_t bid = blockIdx.x;
    if (bid >= lv.first[lv.nlev]) return;
    int li = 0;
    while (bid >= lv.first[li + 1]) ++li;
    const int32_t* __restrict__ slots = lv.slots[li];
    const uint64_t* __restrict__ keys = lv.keys[li];
    const double2* __restrict__ Mh = lv.Mh[li];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int* src = s_src[wave];
    const int nc = lv.ncell[li];
    const int cell0 = static_cast<int>(bid - lv.first[li]) * kUnifCells;
    const int f = blockIdx.y * 64 + lane;
    const int fr = f < NF ? f : 0;
    // the first children among the workgroup's cells
    uint64_t heads;
    {
        const int i = cell0 + lane;
        const bool head = lane < kUnifCells && i < nc && (i == 0 || (keys[i] >> 3) != (keys[i - 1] >> 3));
        heads = __ballot(head);
    }
    for (int turn = 0; heads; ++turn, heads &= heads - 1) {
        if ((turn & 3) != wave) continue;
        const int c0 = cell0 + __builtin_amdgcn_readfirstlane(__builtin_ctzll(heads));
        const uint64_t parent = keys[c0] >> 3;
        int child[8];  // target cells by child index
        uint32_t there = 0;
#pragma unroll
        for (int a = 0; a < 8; ++a) child[a] = -1;
        for (int i = lane; i < 8 * kDirs; i += 64) src[i] = -1;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // the wave's LDS accesses run in order
        for (int c = c0; c < nc && c < c0 + 8 && (keys[c] >> 3) == parent; ++c) {
            const int par = __builtin_amdgcn_readfirstlane(static_cast<int>(keys[c] & 7u));
            there |= 1u << par;
#pragma unroll
            for (int a = 0; a < 8; ++a)
                if (a == par) child[a] = c;
            for (int j = lane; j < kFarSlots; j += 64) {
                const int v = slots[static_cast<int64_t>(c) * kFarSlots + j];
                if (v < 0) continue;
                // offset + target child = 2 direction + source child, per axis
                const int pos = slotpos[par * kFarSlots + j];
                const int tx = pos / 49 - 3 + ((par >> 2) & 1), ty = (pos / 7) % 7 - 3 + ((par >> 1) & 1),
                          tz = pos % 7 - 3 + (par & 1);
                const int dir = (((tx >> 1) + 1) * 3 + (ty >> 1) + 1) * 3 + (tz >> 1) + 1;
                src[8 * dir + ((tx & 1) << 2 | (ty & 1) << 1 | (tz & 1))] = v;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        double2 acc[8];
#pragma unroll
        for (int a = 0; a < 8; ++a) acc[a] = make_double2(0., 0.);
        for (int dir = 0; dir < kDirs; ++dir) {
            const int at = lane < 8 ? src[8 * dir + lane] : -1;
            uint32_t srcs = static_cast<uint32_t>(__ballot(at >= 0));
            if (srcs == 0) continue;  // no source there (nor in the parent itself)
            const int dx = dir / 9 - 1, dy = (dir / 3) % 3 - 1, dz = dir % 3 - 1;
            if constexpr (!FULL) {
#pragma unroll 1
                for (; srcs; srcs &= srcs - 1) {
                    const int b = __builtin_ctz(srcs);
                    const double2 x = Mh[static_cast<int64_t>(__builtin_amdgcn_readlane(at, b)) * NF + fr];
                    double2 k[8];
                    uint32_t far = 0;  // targets that have b among their sources
#pragma unroll
                    for (int a = 0; a < 8; ++a) {
                        if (!(there >> a & 1)) continue;
                        const int px = 2 * dx + ((b >> 2) & 1) - ((a >> 2) & 1), py = 2 * dy + ((b >> 1) & 1) - ((a >> 1) & 1),
                                  pz = 2 * dz + (b & 1) - (a & 1);
                        if (abs(px) <= 1 && abs(py) <= 1 && abs(pz) <= 1) continue;  // near pairs
                        far |= 1u << a;
                        k[a] = K[static_cast<int64_t>(((px + 3) * 7 + py + 3) * 7 + pz + 3) * NF + fr];
                    }
#pragma unroll
                    for (int a = 0; a < 8; ++a) {
                        if (!(far >> a & 1)) continue;
                        acc[a].x = fma(k[a].x, x.x, fma(-k[a].y, x.y, acc[a].x));
                        acc[a].y = fma(k[a].x, x.y, fma(k[a].y, x.x, acc[a].y));
                    }
                }
                continue;
            }
            double2 m[8];
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                const int v = __builtin_amdgcn_readlane(at, b);
                m[b] = v >= 0 ? Mh[static_cast<int64_t>(v) * NF + fr] : make_double2(0., 0.);
            }
#pragma unroll
            for (int ox = -1; ox <= 1; ++ox)
#pragma unroll
                for (int oy = -1; oy <= 1; ++oy)
#pragma unroll
                    for (int oz = -1; oz <= 1; ++oz) {
                        const int px = 2 * dx + ox, py = 2 * dy + oy, pz = 2 * dz + oz;
                        if (abs(px) <= 1 && abs(py) <= 1 && abs(pz) <= 1) continue;  // near pairs
                        const double2 k = K[static_cast<int64_t>(((px + 3) * 7 + py + 3) * 7 + pz + 3) * NF + fr];
#pragma unroll
                        for (int a = 0; a < 8; ++a) {
                            const int bx = ((a >> 2) & 1) + ox, by = ((a >> 1) & 1) + oy, bz = (a & 1) + oz;
                            if (bx < 0 || bx > 1 || by < 0 || by > 1 || bz < 0 || bz > 1) continue;
                            const double2 x = m[bx << 2 | by << 1 | bz];
                            acc[a].x = fma(k.x, x.x, fma(-k.y, x.y, acc[a].x));
                            acc[a].y = fma(k.x, x.y, fma(k.y, x.x, acc[a].y));
                        }
                    }
        }
        const double scale = lv.scale[li];
        if (f < NF) {
#pragma unroll
            for (int a = 0; a < 8; ++a) {
                if (child[a] < 0) continue;
                double2* o = lv.Lh[li] + static_cast<int64_t>(child[a]) * NF + f;
                o->x += scale * acc[a].x;
                o->y += scale * acc[a].y;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // src is rewritten only after these reads
    }
}

#define HFMM_UNIF_ORDERS(X) X(5) X(6) X(7) X(8)

int run_unif_forward(Context* c, int l) {
    const int64_t nc = c->ncell[l];
    if (nc == 0) return HFMM_OK;
    const dim3 grid(static_cast<unsigned>(nc));
    const double* M = c->d_M.as<double>() + c->lvl_off[l] * c->LD;
    double2* Mh = reinterpret_cast<double2*>(c->d_Mt.as<double>() + c->lvl_off[l] * c->glob.k);
    const double2* tw = reinterpret_cast<const double2*>(c->d_utw.as<double>());
    prof_begin(c, "unif_forward");
    switch (c->ops.p) {
#define CASE(PP) case PP: hipLaunchKernelGGL(k_unif_forward<PP>, grid, dim3(64), 0, c->stream, nc, M, c->LD, tw, Mh); break;
        HFMM_UNIF_ORDERS(CASE)
#undef CASE
        default: return fail(c, HFMM_ERR_ARG, "uniform M2L: unsupported order");
    }
    prof_end(c);
    return check_launch(c, "unif_forward");
}

int run_unif_inverse(Context* c, int l) {
    const int64_t nc = c->ncell[l];
    if (nc == 0) return HFMM_OK;
    const dim3 grid(static_cast<unsigned>(nc));
    const double2* Lh = reinterpret_cast<const double2*>(c->d_Lt.as<double>() + c->lvl_off[l] * c->glob.k);
    double* L = c->d_L.as<double>() + c->lvl_off[l] * c->LD;
    const double2* tw = reinterpret_cast<const double2*>(c->d_utw.as<double>());
    prof_begin(c, "unif_inverse");
    switch (c->ops.p) {
#define CASE(PP) case PP: hipLaunchKernelGGL(k_unif_inverse<PP>, grid, dim3(64), 0, c->stream, nc, Lh, tw, L, c->LD); break;
        HFMM_UNIF_ORDERS(CASE)
#undef CASE
        default: return fail(c, HFMM_ERR_ARG, "uniform M2L: unsupported order");
    }
    prof_end(c);
    return check_launch(c, "unif_inverse");
}

int run_unif_m2l(Context* c) {
    const int L = c->height() - 1;
    const int lo = c->work_upper > c->top() ? c->work_upper : c->top();
    const int hi = c->work_lower - 1 < L ? c->work_lower - 1 : L;
    const int k = c->glob.k;
    UnifLevels full{}, few{};  // by the children that the level's parents have
    for (int l = lo; l <= hi; ++l) {
        const int64_t nc = c->ncell[l];
        if (nc == 0) continue;
        const int below = l == c->top() && l < L ? l + 1 : l;  // the top level goes with the one below it
        UnifLevels& lv = c->ncell[below] >= kUnifFull * c->ncell[below - 1] ? full : few;
        const int i = lv.nlev++;
        lv.scale[i] = 2. / (c->P.box_width / static_cast<double>(int64_t(1) << (l - c->set_levels)));
        lv.slots[i] = c->d_m2l.as<int32_t>() + static_cast<size_t>(c->m2l_off[l]) * kFarSlots;
        lv.keys[i] = c->d_cellkey.as<uint64_t>() + c->lvl_off[l];
        lv.Mh[i] = reinterpret_cast<const double2*>(c->d_Mt.as<double>() + c->lvl_off[l] * k);
        lv.Lh[i] = reinterpret_cast<double2*>(c->d_Lt.as<double>() + c->lvl_off[l] * k);
        lv.ncell[i] = static_cast<int>(nc);
        lv.first[i + 1] = lv.first[i] + (nc + kUnifCells - 1) / kUnifCells;
    }
    const int16_t* sp = c->d_slotpos.as<int16_t>();
    const double2* K = reinterpret_cast<const double2*>(c->d_uK.as<double>());
    const int N = 2 * c->ops.p - 1, NF = c->ops.p * N * N;
    const auto grid = [&](const UnifLevels& lv) {
        return dim3(static_cast<unsigned>(lv.first[lv.nlev]), static_cast<unsigned>((NF + 63) / 64));
    };
    prof_begin(c, "unif_m2l");
    switch (c->ops.p) {
#define CASE(PP)                                                                                                          \
    case PP:                                                                                                              \
        if (full.nlev) hipLaunchKernelGGL((k_unif_m2l<PP, true>), grid(full), dim3(256), 0, c->stream, full, sp, K);      \
        if (few.nlev) hipLaunchKernelGGL((k_unif_m2l<PP, false>), grid(few), dim3(256), 0, c->stream, few, sp, K);        \
        break;
        HFMM_UNIF_ORDERS(CASE)
#undef CASE
        default: prof_end(c); return fail(c, HFMM_ERR_ARG, "uniform M2L: unsupported order");
    }
    HFMM_TRY(check_launch(c, "unif_m2l"));
    prof_end(c);
    return HFMM_OK;
}

}  // namespace

int run_global_compress(Context* c, int l) {
    if (c->m2l_scheme == HFMM_M2L_UNIFORM) return run_unif_forward(c, l);
    const int64_t nc = c->ncell[l];
    if (nc == 0) return HFMM_OK;
    const int k = c->glob.k, R = (k + 63) / 64;
    const double* M = c->d_M.as<double>() + c->lvl_off[l] * c->LD;
    double* Mt = c->d_Mt.as<double>() + c->lvl_off[l] * k;
    prof_begin(c, "global_compress");
    const double* Bt = c->d_gBt.as<double>();
    const int nn = c->ops.nn;
    const dim3 grid(static_cast<unsigned>(nc));
    switch (R) {
#define CASE(RR) case RR: hipLaunchKernelGGL(k_global_compress<RR>, grid, dim3(64), 0, c->stream, nc, M, c->LD, Bt, nn, k, Mt); break;
        CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
        default: return fail(c, HFMM_ERR_ARG, "global M2L rank above 512");
    }
    prof_end(c);
    return check_launch(c, "global_compress");
}

int run_global_decompress(Context* c, int l) {
    if (c->m2l_scheme == HFMM_M2L_UNIFORM) return run_unif_inverse(c, l);
    const int64_t nc = c->ncell[l];
    if (nc == 0) return HFMM_OK;
    const int k = c->glob.k;
    prof_begin(c, "global_decompress");
    hipLaunchKernelGGL(k_global_decompress, dim3(static_cast<unsigned>(nc)), dim3(64), 0, c->stream, nc,
                       c->d_Lt.as<double>() + c->lvl_off[l] * k, k, c->d_gU.as<double>(), c->ops.nn,
                       c->d_L.as<double>() + c->lvl_off[l] * c->LD, c->LD);
    prof_end(c);
    return check_launch(c, "global_decompress");
}

// The padded row-major operators of the MFMA M2L, built once per operator set.
static int prepare_global_mfma(Context* c, int KP) {
    if (c->gcr_kp == KP) return HFMM_OK;
    HFMM_TRY(ensure(c, c->d_gCr, sizeof(double) * 343 * static_cast<size_t>(KP) * KP));
    hipLaunchKernelGGL(k_global_pad_ops, dim3(343), dim3(256), 0, c->stream, c->d_gC.as<double>(), c->glob.k, KP,
                       c->d_gCr.as<double>());
    HFMM_TRY(check_launch(c, "global_pad_ops"));
    c->gcr_kp = KP;
    return HFMM_OK;
}

int run_global_m2l(Context* c) {
    if (c->m2l_scheme == HFMM_M2L_UNIFORM) return run_unif_m2l(c);
    const int k = c->glob.k, R = (k + 63) / 64;
    if (R > kMaxRankRows) return fail(c, HFMM_ERR_ARG, "global M2L rank above 512");
    const int NR = (k + 15) / 16;
    if (NR <= kGlobalMfmaMaxTiles) {
        HFMM_TRY(prepare_global_mfma(c, 16 * NR));
        HFMM_TRY(ensure_parity_order(c));
        int tiles = 0;
        const M2LLevels lv = make_levels(c, 16, tiles);
        if (tiles == 0) return HFMM_OK;
        prof_begin(c, "global_m2l");
        const dim3 grid(static_cast<unsigned>(tiles));
        const int32_t* slots = c->d_m2l.as<int32_t>();
        const int32_t* ord = c->d_order.as<int32_t>();
        const int32_t* pc = c->d_pcount.as<int32_t>();
        const int16_t* sp = c->d_slotpos.as<int16_t>();
        const double* Cr = c->d_gCr.as<double>();
        const double* Mt = c->d_Mt.as<double>();
        double* Lt = c->d_Lt.as<double>();
        switch (NR) {
#define CASE(N) case N: hipLaunchKernelGGL(k_global_m2l_mfma<N>, grid, dim3(256), 0, c->stream, lv, slots, ord, pc, sp, Cr, Mt, k, Lt); break;
            CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
            CASE(9) CASE(10) CASE(11) CASE(12) CASE(13) CASE(14) CASE(15) CASE(16)
#undef CASE
            default: break;
        }
        prof_end(c);
        return check_launch(c, "global_m2l");
    }
    const int L = c->height() - 1;
    // the M2L levels of the working range, from the top
    const int lo = c->work_upper > c->top() ? c->work_upper : c->top();
    const int hi = c->work_lower - 1 < L ? c->work_lower - 1 : L;
    prof_begin(c, "global_m2l");
    for (int l = lo; l <= hi; ++l) {
        const int64_t nc = c->ncell[l];
        if (nc == 0) continue;
        const double scale = 2. / (c->P.box_width / static_cast<double>(int64_t(1) << (l - c->set_levels)));
        const int32_t* slots = c->d_m2l.as<int32_t>() + static_cast<size_t>(c->m2l_off[l]) * kFarSlots;
        const uint64_t* keys = c->d_cellkey.as<uint64_t>() + c->lvl_off[l];
        const double* Mt = c->d_Mt.as<double>() + c->lvl_off[l] * k;
        double* Lt = c->d_Lt.as<double>() + c->lvl_off[l] * k;
        const int16_t* sp = c->d_slotpos.as<int16_t>();
        const double* Cg = c->d_gC.as<double>();
        const dim3 grid(static_cast<unsigned>(nc));
        switch (R) {
#define CASE(RR) case RR: hipLaunchKernelGGL(k_global_m2l<RR>, grid, dim3(64), 0, c->stream, nc, slots, keys, sp, Cg, Mt, k, scale, Lt); break;
            CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
            default: break;
        }
        HFMM_TRY(check_launch(c, "global_m2l"));
    }
    prof_end(c);
    return HFMM_OK;
}

}  // namespace hfmm

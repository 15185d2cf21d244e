// m2l_f64.hip -- the symmetric scheme's M2L in FP64
// (Src/Kernels/Chebyshev/FChebSymKernel.hpp:210-328): for every far-field pair
// (target t, source s at relative position pos, canonical operator c)
//   L_t += 2/w U_c[pv] (V_c[pv]^T M_s)
// as two dense products on v_mfma_f64_16x16x4f64 with the compressed
// expansions C in device memory between them.
//
// Positions that differ only in the signs of their coordinates share one
// operator up to a reflection of the nodes, pv(pos)[n] = pv(|pos|)[R n].
// Split into even and odd parts along each axis (8 classes of about p^3/8
// half-nodes), V^T R M is a sum of the 8 class products with signs:
//   C_sigma = sum_k (-1)^|k & sigma| V_k^T M_k,   k, sigma in {0..7}
// so the products of the 56 offsets |pos| serve all 189 positions of a cell:
// the 8 signed sums are an 8-point Hadamard transform.  Transposed, a target's
// locals are sum_{|pos|} U_k (sum_sigma (-1)^|k & sigma| C_sigma) per class.
// A product per cell takes p^3 sum(rank over 56) FMAs instead of p^3 sum(rank
// over 189) (3.55 times fewer at order 7), and the ranks of all offsets lie in
// one row index, padded to multiples of 4 instead of 16 (1396 rows for 1331 at
// order 7; one operator at a time padded them to 6464 for 4719).
//
//   k_m2l_up    per tile of 16 C cells as sources: the class products of every
//               row, the Hadamard sums, and each sum to the cell it is for:
//               C[target][row block][|pos|][variant][row]
//   k_m2l_down  per tile of 16 C cells as targets: their own C, streamed, the
//               Hadamard sums, the class products, the locals
//
// Both run one class per wave (8 waves): wave w and w + 4 share a SIMD, so the
// classes are dealt to give every SIMD the same number of MFMAs (order 7: 23,
// 21, 21, 21 per 16 rows).  A step is 32 (row, cell) lines of 16; the tile that
// holds the Hadamard operands is double buffered, one barrier per step.
//
// Of the SIMD cycles, MFMAs take 43% upward and 59% downward (1M uniform, h7, order
// 7), VALU instructions 11% and 16% more: the two do not overlap (4 VALU
// instructions beside a 66-cycle FP64 MFMA add 16 cycles).  The rest is waiting:
// one workgroup of 8 waves fits a CU at orders 7 and 8 and has a barrier per step,
// and upward every thread masks and stores 8 sums of 8 bytes per step.  1M uniform
// particles, h7, order 7: 55.7 (one operator per slot) -> 15.8 ms, 33.9 TFLOP/s
// executed; 10M Plummer, h8, order 8: 202 -> 42 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <vector>

#include "fmm_common.hpp"
#include "hfmm_internal.hpp"
#include "m2l_plan.hpp"

namespace hfmm {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kTauStride = 60; // bytes per cell of a table over the offsets (whole words)
constexpr int kMWaves = 8;
constexpr int kMThreads = 64 * kMWaves;
constexpr int kMaxSteps = 256;  // row blocks: 56 offsets of rank <= 64
constexpr int kTgtRow = 8 * (kTau + 1) + 4;  // entries of a source in the table of its targets (rows on other banks)
constexpr int kXcdChunk = 16;   // consecutive tiles that run on one XCD

// Keeps the scheduler from moving the work of a phase between the MFMAs of another.
#define M2L_FENCE __builtin_amdgcn_sched_barrier(0)

// Wave -> class (bit a: odd along axis a).
__host__ __device__ constexpr int class_of(int w) {
    return w == 0 ? 0 : w == 1 ? 1 : w == 2 ? 2 : w == 3 ? 4 : w == 4 ? 7 : w == 5 ? 3 : w == 6 ? 5 : 6;
}
__host__ __device__ constexpr int wave_of(int k) {
    return k == 0 ? 0 : k == 1 ? 1 : k == 2 ? 2 : k == 4 ? 3 : k == 7 ? 4 : k == 3 ? 5 : k == 5 ? 6 : 7;
}
__host__ __device__ constexpr int odd_axes(int k) { return (k & 1) + ((k >> 1) & 1) + ((k >> 2) & 1); }

template <int P>
struct Cls {
    static constexpr int HE = (P + 1) / 2, HO = P / 2;  // even / odd half-nodes per axis
    static constexpr int kH3 = HE * HE * HE;
    static constexpr int kItems = (kH3 * 16 + kMThreads - 1) / kMThreads;  // half-nodes of 16 cells per thread
    __host__ __device__ static constexpr int side(int k, int a) { return (k >> a) & 1 ? HO : HE; }
    // half-nodes of a class with o odd axes, MFMA K steps (4 half-nodes), row tiles (16)
    __host__ __device__ static constexpr int size(int o) {
        int s = 1;
        for (int a = 0; a < 3; ++a) s *= a < o ? HO : HE;
        return s;
    }
    __host__ __device__ static constexpr int ks(int o) { return (size(o) + 3) / 4; }
    __host__ __device__ static constexpr int ksp(int o) { return (ks(o) + 1) / 2; }  // pairs of K steps
    __host__ __device__ static constexpr int nt(int o) { return (size(o) + 15) / 16; }
    // operator doubles of one row block before wave w: up (K = half-nodes) and down (M = half-nodes)
    __host__ __device__ static constexpr int up_off(int w) {
        int s = 0;
        for (int v = 0; v < w; ++v) s += 128 * ksp(odd_axes(class_of(v)));
        return s;
    }
    __host__ __device__ static constexpr int down_off(int w) {
        int s = 0;
        for (int v = 0; v < w; ++v) s += 256 * nt(odd_axes(class_of(v)));
        return s;
    }
    // LDS doubles of the class expansions of 16 cells before wave w
    __host__ __device__ static constexpr int exp_off(int w) {
        int s = 0;
        for (int v = 0; v < w; ++v) s += 64 * ks(odd_axes(class_of(v)));
        return s;
    }
    // LDS rows of the locals' classes before wave w
    __host__ __device__ static constexpr int loc_off(int w) {
        int s = 0;
        for (int v = 0; v < w; ++v) s += 16 * nt(odd_axes(class_of(v)));
        return s;
    }
};

struct M2LArgs {
    M2LLevels lv;
    int64_t first, ncell;  // cells of the working levels
    int rb0, rb1;          // row blocks of this launch
    uint32_t off0, stride;  // C bytes before rb0, and C bytes per target
    const int32_t* slots;
    const uint64_t* keys;
    const RowInfo* rows;
    const uint16_t* slot_tau;  // [8][189] 8 offset + sigma of a target's slot, then the same seen from the other cell
    const double* ops;         // fragments, row block by row block
    double* C;
    double* acc;               // partial locals between launches over parts of the rows
    int load, store;           // continue from acc / leave the partial sums there
};

__device__ __forceinline__ int tile_of(int bid) {
    const int q = bid / (8 * kXcdChunk), r = bid % (8 * kXcdChunk);
    return q * 8 * kXcdChunk + (r & 7) * kXcdChunk + (r >> 3);
}

__device__ __forceinline__ int level_of(const M2LLevels& lv, int64_t cell) {
    int li = 0;
    while (li + 1 < lv.nlev && cell >= lv.cell_off[li + 1]) ++li;
    return li;
}

__device__ __forceinline__ void hadamard8(double (&d)[8]) {
#pragma unroll
    for (int b = 1; b < 8; b <<= 1)
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (!(i & b)) {
                const double u = d[i], v = d[i | b];
                d[i] = u + v;
                d[i | b] = u - v;
            }
}

// Buffer accesses for the masked reads and writes of C: past the buffer's end a
// store is dropped and a load gives 0, so a lane without a partner takes part
// with the offset kNowhere.  A branch around each access would hide their number
// from the wait counts: every wait for operators would wait for all stores.

typedef uint32_t u2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(double* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(p, 0, static_cast<int>(bytes), 0x00027000);
}
__device__ __forceinline__ double buffer_load(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, static_cast<int>(off), 0, 0));
}
__device__ __forceinline__ void buffer_store(__amdgpu_buffer_rsrc_t r, uint32_t off, double v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, static_cast<int>(off), 0, 0);
}

// Bytes into a target's C of the 8 signs of a row.
__device__ __forceinline__ void variant_offsets(const RowInfo& r, uint32_t off0, uint32_t (&at)[8]) {
    at[0] = r.off - off0;
    at[1] = at[0] + r.sign[0];
#pragma unroll
    for (int s = 0; s < 2; ++s) at[2 + s] = at[s] + r.sign[1];
#pragma unroll
    for (int s = 0; s < 4; ++s) at[4 + s] = at[s] + r.sign[2];
}

// The steps (RB row blocks each) of [rb0, rb1) that hold a flagged offset, in
// ascending order, as step numbers relative to rb0; called by every thread.
template <int RB>
__device__ __forceinline__ int active_steps(const M2LArgs& a, const int* s_flag, uint16_t* s_list,
                                            int* s_count) {
    const int nst = (a.rb1 - a.rb0 + RB - 1) / RB;
    if (threadIdx.x < 64) {
        int n = 0;
        for (int b = 0; b < nst; b += 64) {
            const int st = b + static_cast<int>(threadIdx.x);
            bool on = false;
            if (st < nst) {
                const int r0 = 16 * (a.rb0 + RB * st);
                const int r1 = min(r0 + 16 * RB, 16 * a.rb1) - 1;
                const int t0 = a.rows[r0].tau, t1 = a.rows[r1].tau;
                for (int t = t0; t <= t1; ++t) on |= s_flag[t] != 0;
            }
            const uint64_t m = __ballot(on);
            if (on) s_list[n + __popcll(m & ((1ull << threadIdx.x) - 1ull))] = static_cast<uint16_t>(st);
            n += __popcll(m);
        }
        if (threadIdx.x == 0) *s_count = n;
    }
    __syncthreads();
    return *s_count;
}

// LDS of a launch: the tile buffers, then the tables.
template <int C>
struct Lds {
    static constexpr int RB = 2 / C;
    static constexpr int kRow = 16 * RB + 2;             // padded rows of one (class, cell) line
    static constexpr int kBuf = kMWaves * 16 * C * kRow;  // doubles of one tile
};

struct SmemLayout {
    int cells, rows, flags, bytes;  // byte offsets
};
inline SmemLayout smem_layout(int big_doubles, int cell_bytes, int nrows) {
    SmemLayout s;
    s.cells = big_doubles * 8;
    s.rows = s.cells + ((cell_bytes + 15) & ~15);
    s.flags = s.rows + nrows * static_cast<int>(sizeof(RowInfo));
    s.bytes = s.flags + 4 * (kTau + 2 + 2) + 2 * kMaxSteps;
    return s;
}

// ---------------------------------------------------------------------------
template <int P, int C, int O, bool WIDE>
__device__ __forceinline__ void up_body(const M2LArgs& a, const SmemLayout& sl, char* smem,
                                        double (&nodes)[C][Cls<P>::kItems][8], int wave) {
    using K = Cls<P>;
    constexpr int RB = Lds<C>::RB, KROW = Lds<C>::kRow, BUF = Lds<C>::kBuf;
    constexpr int KS = K::ks(O), KSP = K::ksp(O);
    double* big = reinterpret_cast<double*>(smem);
    const uint32_t* s_tgt = reinterpret_cast<const uint32_t*>(smem + sl.cells);
    int* s_flag = reinterpret_cast<int*>(smem + sl.flags);
    int* s_count = s_flag + kTau + 2;
    uint16_t* s_list = reinterpret_cast<uint16_t*>(s_flag + kTau + 4);
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, kq = lane >> 4;

    // class expansions of the 16 C cells, one column tile at a time
    double b[C][KS];
#pragma unroll
    for (int c = 0; c < C; ++c) {
#pragma unroll
        for (int it = 0; it < K::kItems; ++it) {
            const int e = tid + it * kMThreads;
            if (K::kH3 * 16 % kMThreads && e >= K::kH3 * 16) break;
            const int h = e % K::kH3, cc = e / K::kH3;
            const int hx = h % K::HE, hy = (h / K::HE) % K::HE, hz = h / (K::HE * K::HE);
            double(&d)[8] = nodes[c][it];
            hadamard8(d);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if (hx >= K::side(k, 0) || hy >= K::side(k, 1) || hz >= K::side(k, 2)) continue;
                const int m = (hz * K::side(k, 1) + hy) * K::side(k, 0) + hx;
                big[K::exp_off(wave_of(k)) + (m >> 2) * 64 + 16 * (m & 3) + cc] = d[k];
            }
        }
        // the fill of the last K step of each class
#pragma unroll
        for (int w = 0; w < kMWaves; ++w) {
            const int sz = K::size(odd_axes(class_of(w))), k4 = 4 * K::ks(odd_axes(class_of(w)));
            for (int e = tid; e < (k4 - sz) * 16; e += kMThreads) {
                const int m = sz + e / 16;
                big[K::exp_off(w) + (m >> 2) * 64 + 16 * (m & 3) + e % 16] = 0.;
            }
        }
        __syncthreads();
        const double* mine = big + K::exp_off(0) + lane;
        int off = 0;
        for (int v = 0; v < wave; ++v) off += 64 * K::ks(odd_axes(class_of(v)));
#pragma unroll
        for (int s = 0; s < KS; ++s) b[c][s] = mine[off + 64 * s];
        __syncthreads();
    }
    const int nact = active_steps<RB>(a, s_flag, s_list, s_count);
    if (nact == 0) return;

    int wop = 0, rbd = 0;
#pragma unroll
    for (int v = 0; v < kMWaves; ++v) {
        const int d = 128 * K::ksp(odd_axes(class_of(v)));
        if (v < wave) wop += d;
        rbd += d;
    }
    const double2* ops = reinterpret_cast<const double2*>(a.ops + static_cast<int64_t>(a.rb0) * rbd + wop) + lane;
    // this thread's line of a step's Hadamard sums
    const int erow = tid % (16 * RB), ecol = tid / (16 * RB);
    const uint32_t* etg = s_tgt + ecol * kTgtRow;
    const __amdgpu_buffer_rsrc_t out = buffer_of(a.C, static_cast<uint32_t>(a.stride * a.ncell));

    auto fetch = [&](int st, double2 (&o)[RB][KSP]) {
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int s = 0; s < KSP; ++s) o[r][s] = ops[static_cast<int64_t>(st * RB + r) * (rbd / 2) + 64 * s];
    };
    // quarter q of the step's MFMAs, the two accumulators in turn
    auto products = [&](int q, const double2 (&av)[RB][KSP], d4 (&acc)[RB][C]) {
#pragma unroll
        for (int s = (KS * q) / 4; s < (KS * (q + 1)) / 4; ++s)
#pragma unroll
            for (int r = 0; r < RB; ++r)
#pragma unroll
                for (int c = 0; c < C; ++c)
                    acc[r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(s & 1 ? av[r][s / 2].y : av[r][s / 2].x, b[c][s],
                                                                     acc[r][c], 0, 0, 0);
    };
    auto clear = [&](d4 (&acc)[RB][C]) {
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int c = 0; c < C; ++c) acc[r][c] = d4{0., 0., 0., 0.};
    };
    auto keep = [&](int buf, const d4 (&acc)[RB][C]) {
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int c = 0; c < C; ++c) {
                double2* d = reinterpret_cast<double2*>(big + buf * BUF + (wave * 16 * C + 16 * c + col) * KROW + 16 * r +
                                                        4 * kq);
                d[0] = make_double2(acc[r][c][0], acc[r][c][1]);
                d[1] = make_double2(acc[r][c][2], acc[r][c][3]);
            }
    };
    // the sums of a step in three parts, between the MFMAs of the next
    double d[8];
    const RowInfo* rows = reinterpret_cast<const RowInfo*>(smem + sl.rows) + erow;
    RowInfo ri;
    uint32_t tg[8];
    auto send_read = [&](int buf, int st) {
        ri = rows[16 * RB * st];
#pragma unroll
        for (int k = 0; k < 8; ++k) d[k] = big[buf * BUF + (wave_of(k) * 16 * C + ecol) * KROW + erow];
    };
    auto send_sum = [&]() {
        const uint4* t = reinterpret_cast<const uint4*>(etg + 8 * ri.tau);
        const uint4 lo = t[0], hi = t[1];
        tg[0] = lo.x, tg[1] = lo.y, tg[2] = lo.z, tg[3] = lo.w;
        tg[4] = hi.x, tg[5] = hi.y, tg[6] = hi.z, tg[7] = hi.w;
        hadamard8(d);
    };
    auto send_store = [&]() {
        uint32_t at[8];
        variant_offsets(ri, a.off0, at);
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            if constexpr (WIDE) {  // tg: the target itself
                if (tg[s] != kNowhere)
                    *reinterpret_cast<double*>(reinterpret_cast<char*>(a.C) + static_cast<uint64_t>(tg[s]) * a.stride + at[s]) = d[s];
            } else {
                buffer_store(out, tg[s] + at[s], d[s]);
            }
        }
    };
    // operators of the next step, this step's products, the last step's sums
    auto step = [&](int i, const double2 (&av)[RB][KSP], double2 (&nv)[RB][KSP]) {
        d4 acc[RB][C];
        fetch(s_list[i + 1 < nact ? i + 1 : i], nv);
        send_read((i - 1) & 1, s_list[i - 1]);
        clear(acc);
        M2L_FENCE;
        products(0, av, acc);
        M2L_FENCE;
        send_sum();
        M2L_FENCE;
        products(1, av, acc);
        M2L_FENCE;
        send_store();
        M2L_FENCE;
        products(2, av, acc);
        products(3, av, acc);
        keep(i & 1, acc);
        __syncthreads();
    };
    double2 ev[RB][KSP], ov[RB][KSP];
    fetch(s_list[0], ev);
    fetch(s_list[nact > 1 ? 1 : 0], ov);
    {
        d4 acc[RB][C];
        clear(acc);
#pragma unroll
        for (int q = 0; q < 4; ++q) products(q, ev, acc);
        keep(0, acc);
    }
    __syncthreads();
    int i = 1;
    for (; i + 1 < nact; i += 2) {
        step(i, ov, ev);
        step(i + 1, ev, ov);
    }
    if (i < nact) step(i, ov, ev);
    send_read((nact - 1) & 1, s_list[nact - 1]);
    send_sum();
    send_store();
}

// The slots of a tile's cells, kSlotItems per thread (the cells' rows are
// contiguous), -1 past the last cell.
template <int C>
struct TileSlots {
    static constexpr int kSlotItems = (16 * C * kFarSlots + kMThreads - 1) / kMThreads;
    int32_t t[kSlotItems];
    __device__ __forceinline__ void load(const M2LArgs& a, int64_t cell0, int ncol) {
        const int32_t* g = a.slots + cell0 * kFarSlots;
#pragma unroll
        for (int i = 0; i < kSlotItems; ++i) {
            const int e = static_cast<int>(threadIdx.x) + i * kMThreads;
            t[i] = e < ncol * kFarSlots ? g[e] : -1;
        }
    }
    // f(cell of the tile, 8 offset + sigma, slot value) for every slot that is taken
    template <class F>
    __device__ __forceinline__ void each(const uint16_t* s_slot, const int* s_par, F f) const {
#pragma unroll
        for (int i = 0; i < kSlotItems; ++i) {
            if (t[i] < 0) continue;
            const int e = static_cast<int>(threadIdx.x) + i * kMThreads;
            const int cc = e / kFarSlots, j = e - cc * kFarSlots;
            f(cc, static_cast<int>(s_slot[s_par[cc] * kFarSlots + j]), t[i]);
        }
    }
};

// The slots' table (dir 0: positions seen from the cell, 1:
// from the other cell), the parities and the
// first cells of the levels of the tile's cells into the LDS.
struct TileTables {
    uint16_t* slot;  // at the end of the tile buffers, free before the first step
    int* par;
    int* first;
    int* flag;
};
template <int C>
__device__ __forceinline__ TileTables load_tables(const M2LArgs& a, const SmemLayout& sl, char* smem, int dir, int64_t cell0,
                                                  int ncol) {
    TileTables t;
    t.slot = reinterpret_cast<uint16_t*>(smem + sl.cells) - 8 * kFarSlots;
    t.par = reinterpret_cast<int*>(t.slot) - 32;
    t.first = t.par - 32;
    t.flag = reinterpret_cast<int*>(smem + sl.flags);
    const uint32_t* st = reinterpret_cast<const uint32_t*>(a.slot_tau + dir * 8 * kFarSlots);
    for (int i = threadIdx.x; i < 4 * kFarSlots; i += kMThreads) reinterpret_cast<uint32_t*>(t.slot)[i] = st[i];
    if (threadIdx.x < kTau + 2) t.flag[threadIdx.x] = 0;
    if (static_cast<int>(threadIdx.x) < ncol) {
        const int64_t cell = cell0 + threadIdx.x;
        t.par[threadIdx.x] = static_cast<int>(a.keys[cell] & 7u);
        t.first[threadIdx.x] = static_cast<int>(a.lv.cell_off[level_of(a.lv, cell)] - a.first);
    }
    return t;
}

template <int P, int C, bool WIDE>
__global__ __launch_bounds__(kMThreads, 2) void k_m2l_up(M2LArgs a, SmemLayout sl, const double* __restrict__ M, int LD) {
    extern __shared__ double2 smem_up[];
    char* smem = reinterpret_cast<char*>(smem_up);
    const int64_t cell0 = a.first + static_cast<int64_t>(tile_of(blockIdx.x)) * 16 * C;
    const int64_t end = a.first + a.ncell;
    if (cell0 >= end) return;  // the same for the whole workgroup
    const int ncol = static_cast<int>(min(static_cast<int64_t>(16 * C), end - cell0));
    // every load of the prologue on its way at once
    using K = Cls<P>;
    TileSlots<C> ts;
    ts.load(a, cell0, ncol);
    double nodes[C][K::kItems][8];
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int it = 0; it < K::kItems; ++it) {
            const int e = static_cast<int>(threadIdx.x) + it * kMThreads;
            const int h = e % K::kH3, cc = 16 * c + e / K::kH3;
            const int hx = h % K::HE, hy = (h / K::HE) % K::HE, hz = h / (K::HE * K::HE);
            const bool in = cc < ncol && e < K::kH3 * 16;
            const double* m = M + (cell0 + (in ? cc : 0)) * LD;
#pragma unroll
            for (int f = 0; f < 8; ++f) {
                // a middle node (odd order) has no mirror image
                const bool mid = ((f & 1) && hx == K::HO) || ((f & 2) && hy == K::HO) || ((f & 4) && hz == K::HO);
                const int nx = f & 1 ? P - 1 - hx : hx, ny = f & 2 ? P - 1 - hy : hy, nz = f & 4 ? P - 1 - hz : hz;
                const double v = m[(nz * P + ny) * P + nx];
                nodes[c][it][f] = in && !mid ? v : 0.;
            }
        }
    const TileTables tt = load_tables<C>(a, sl, smem, 1, cell0, ncol);
    for (int i = threadIdx.x; i < 16 * (a.rb1 - a.rb0); i += kMThreads)
        reinterpret_cast<uint4*>(smem + sl.rows)[i] = reinterpret_cast<const uint4*>(a.rows + 16 * static_cast<int64_t>(a.rb0))[i];
    // targets of every source by (offset, sigma): where their C begins
    uint32_t* s_tgt = reinterpret_cast<uint32_t*>(smem + sl.cells);
    for (int e = threadIdx.x; e < 4 * C * kTgtRow; e += kMThreads)
        reinterpret_cast<uint4*>(s_tgt)[e] = make_uint4(kNowhere, kNowhere, kNowhere, kNowhere);
    __syncthreads();
    ts.each(tt.slot, tt.par, [&](int cc, int w, int t) {
        const uint32_t to = static_cast<uint32_t>(tt.first[cc] + t);
        s_tgt[cc * kTgtRow + w] = WIDE ? to : to * a.stride;
        tt.flag[w >> 3] = 1;
    });
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if constexpr (P % 2 == 0) {
        up_body<P, C, 0, WIDE>(a, sl, smem, nodes, wave);
    } else {
        switch (odd_axes(class_of(wave))) {
            case 0: up_body<P, C, 0, WIDE>(a, sl, smem, nodes, wave); break;
            case 1: up_body<P, C, 1, WIDE>(a, sl, smem, nodes, wave); break;
            case 2: up_body<P, C, 2, WIDE>(a, sl, smem, nodes, wave); break;
            default: up_body<P, C, 3, WIDE>(a, sl, smem, nodes, wave); break;
        }
    }
}

// ---------------------------------------------------------------------------
template <int P, int C, int O>
__device__ __forceinline__ void down_body(const M2LArgs& a, const SmemLayout& sl, char* smem, double* __restrict__ L,
                                          int LD, int wave, int tile, int64_t cell0, int ncol) {
    using K = Cls<P>;
    constexpr int RB = Lds<C>::RB, KROW = Lds<C>::kRow, BUF = Lds<C>::kBuf;
    constexpr int NT = K::nt(O);
    double* big = reinterpret_cast<double*>(smem);
    const uint8_t* s_ex = reinterpret_cast<const uint8_t*>(smem + sl.cells);
    int* s_flag = reinterpret_cast<int*>(smem + sl.flags);
    int* s_count = s_flag + kTau + 2;
    uint16_t* s_list = reinterpret_cast<uint16_t*>(s_flag + kTau + 4);
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, kq = lane >> 4;
    const int nact = active_steps<RB>(a, s_flag, s_list, s_count);

    int wop = 0, rbd = 0, lrow = 0;
#pragma unroll
    for (int v = 0; v < kMWaves; ++v) {
        const int n = K::nt(odd_axes(class_of(v)));
        if (v < wave) wop += 256 * n, lrow += 16 * n;
        rbd += 256 * n;
    }
    const double2* ops = reinterpret_cast<const double2*>(a.ops + static_cast<int64_t>(a.rb0) * rbd + wop) + lane;
    d4* part = reinterpret_cast<d4*>(a.acc) + (static_cast<int64_t>(tile) * kMWaves + wave) * K::nt(0) * C * 64 + lane;
    d4 acc[NT][C];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int c = 0; c < C; ++c) acc[t][c] = a.load ? part[(t * C + c) * 64] : d4{0., 0., 0., 0.};

    const int erow = tid % (16 * RB), ecol = tid / (16 * RB);
    // the C of the tile's targets
    const __amdgpu_buffer_rsrc_t in =
        buffer_of(reinterpret_cast<double*>(reinterpret_cast<char*>(a.C) + (cell0 - a.first) * a.stride), a.stride * ncol);
    const uint32_t mine = a.off0 - ecol * a.stride;
    const RowInfo* rows = a.rows + 16 * a.rb0 + erow;
    auto fetch = [&](const RowInfo& ri, double (&d)[8]) {
        const int none = ~static_cast<int>(s_ex[ecol * kTauStride + ri.tau]);
        uint32_t at[8];
        variant_offsets(ri, mine, at);
#pragma unroll
        for (int s = 0; s < 8; ++s)  // past every end, where there is no source
            d[s] = buffer_load(in, at[s] | (static_cast<uint32_t>(__builtin_amdgcn_sbfe(none, s, 1)) & 0xFFFFFFF0u));
    };
    auto sums = [&](int buf, double (&d)[8]) {
        hadamard8(d);
#pragma unroll
        for (int k = 0; k < 8; ++k) big[buf * BUF + (wave_of(k) * 16 * C + ecol) * KROW + erow] = d[k];
    };
    auto operators = [&](int st, double2 (&o)[RB][NT][2]) {
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int h = 0; h < 2; ++h) o[r][t][h] = ops[static_cast<int64_t>(st * RB + r) * (rbd / 2) + (2 * t + h) * 64];
    };
    // operators of the next step and C of the one after it on their way during
    // this step's products, the next step's sums between them
    RowInfo rn;  // of the next C to fetch
    auto step = [&](int i, const double2 (&av)[RB][NT][2], double2 (&nv)[RB][NT][2], double (&d)[8]) {
        double2 bv[RB][C][2];
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const double2* x = reinterpret_cast<const double2*>(
                    big + (i & 1) * BUF + (wave * 16 * C + 16 * c + col) * KROW + 16 * r + 4 * kq);
                bv[r][c][0] = x[0];
                bv[r][c][1] = x[1];
            }
        // quarter q of the step's K steps, row block by row block: both tile shapes
        // add a target's terms in the same order (equal bits whatever the shape)
        auto products = [&](int q) {
#pragma unroll
            for (int k = RB * q; k < RB * (q + 1); ++k) {
                const int r = k / 4, s = k % 4;
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int c = 0; c < C; ++c)
                        acc[t][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                            s & 1 ? av[r][t][s / 2].y : av[r][t][s / 2].x,
                            s & 1 ? bv[r][c][s / 2].y : bv[r][c][s / 2].x, acc[t][c], 0, 0, 0);
            }
        };
        operators(s_list[i + 1 < nact ? i + 1 : i], nv);
        M2L_FENCE;
        products(0);
        M2L_FENCE;
        sums((i + 1) & 1, d);
        M2L_FENCE;
        products(1);
        M2L_FENCE;
        fetch(rn, d);
        rn = rows[16 * RB * s_list[i + 3 < nact ? i + 3 : i]];
        M2L_FENCE;
        products(2);
        products(3);
        __syncthreads();
    };
    if (nact > 0) {
        double d[8];
        double2 ev[RB][NT][2], ov[RB][NT][2];
        rn = rows[16 * RB * s_list[0]];
        fetch(rn, d);
        operators(s_list[0], ev);
        rn = rows[16 * RB * s_list[nact > 1 ? 1 : 0]];
        sums(0, d);
        fetch(rn, d);
        rn = rows[16 * RB * s_list[nact > 2 ? 2 : 0]];
        __syncthreads();
        int i = 0;
        for (; i + 1 < nact; i += 2) {
            step(i, ev, ov, d);
            step(i + 1, ov, ev, d);
        }
        if (i < nact) step(i, ev, ov, d);
    }
    if (a.store) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int c = 0; c < C; ++c) part[(t * C + c) * 64] = acc[t][c];
        return;
    }
    // the classes back to nodes, one column tile at a time
#pragma unroll
    for (int c = 0; c < C; ++c) {
        if (c) __syncthreads();
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) big[(lrow + 16 * t + 4 * r + kq) * 17 + col] = acc[t][c][r];
        __syncthreads();
        for (int e = tid; e < K::kH3 * 16; e += kMThreads) {
            const int h = e % K::kH3, cc = e / K::kH3;
            if (16 * c + cc >= ncol) continue;
            const int hx = h % K::HE, hy = (h / K::HE) % K::HE, hz = h / (K::HE * K::HE);
            double d[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const bool in = hx < K::side(k, 0) && hy < K::side(k, 1) && hz < K::side(k, 2);
                const int m = in ? (hz * K::side(k, 1) + hy) * K::side(k, 0) + hx : 0;
                d[k] = in ? big[(K::loc_off(wave_of(k)) + m) * 17 + cc] : 0.;
            }
            hadamard8(d);
            const int64_t cell = cell0 + 16 * c + cc;
            const double scale = a.lv.scale[level_of(a.lv, cell)];
            double* out = L + cell * LD;
#pragma unroll
            for (int f = 0; f < 8; ++f) {
                const bool mid = ((f & 1) && hx == K::HO) || ((f & 2) && hy == K::HO) || ((f & 4) && hz == K::HO);
                if (mid) continue;
                const int nx = f & 1 ? P - 1 - hx : hx, ny = f & 2 ? P - 1 - hy : hy, nz = f & 4 ? P - 1 - hz : hz;
                out[(nz * P + ny) * P + nx] = scale * d[f];
            }
        }
    }
}

template <int P, int C>
__global__ __launch_bounds__(kMThreads, 2) void k_m2l_down(M2LArgs a, SmemLayout sl, double* __restrict__ L, int LD) {
    extern __shared__ double2 smem_down[];
    char* smem = reinterpret_cast<char*>(smem_down);
    const int tile = tile_of(blockIdx.x);
    const int64_t cell0 = a.first + static_cast<int64_t>(tile) * 16 * C;
    const int64_t end = a.first + a.ncell;
    if (cell0 >= end) return;
    const int ncol = static_cast<int>(min(static_cast<int64_t>(16 * C), end - cell0));
    TileSlots<C> ts;
    ts.load(a, cell0, ncol);
    const TileTables tt = load_tables<C>(a, sl, smem, 0, cell0, ncol);
    // signs of each offset that a target has a source at: a byte per (target,
    // offset, sigma) in the tile buffers, then packed to a bit each
    uint64_t* s_at = reinterpret_cast<uint64_t*>(smem);
    for (int i = threadIdx.x; i < 16 * C * kTauStride; i += kMThreads) s_at[i] = 0ull;
    __syncthreads();
    ts.each(tt.slot, tt.par, [&](int cc, int w, int) {
        reinterpret_cast<uint8_t*>(s_at)[cc * 8 * kTauStride + w] = 1;
        tt.flag[w >> 3] = 1;
    });
    __syncthreads();
    uint8_t* s_ex = reinterpret_cast<uint8_t*>(smem + sl.cells);
    for (int i = threadIdx.x; i < 16 * C * kTauStride; i += kMThreads)
        s_ex[i] = static_cast<uint8_t>((s_at[i] * 0x0102040810204080ull) >> 56);  // byte k (0 or 1) -> bit k
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if constexpr (P % 2 == 0) {
        down_body<P, C, 0>(a, sl, smem, L, LD, wave, tile, cell0, ncol);
    } else {
        switch (odd_axes(class_of(wave))) {
            case 0: down_body<P, C, 0>(a, sl, smem, L, LD, wave, tile, cell0, ncol); break;
            case 1: down_body<P, C, 1>(a, sl, smem, L, LD, wave, tile, cell0, ncol); break;
            case 2: down_body<P, C, 2>(a, sl, smem, L, LD, wave, tile, cell0, ncol); break;
            default: down_body<P, C, 3>(a, sl, smem, L, LD, wave, tile, cell0, ncol); break;
        }
    }
}

// ---------------------------------------------------------------------------
// Operator fragments.  Entry of class k, half-node (hx, hy, hz), row (tau, r):
// the mean over the mirror images of the node, with the class's signs, of
// V_c[pv(|pos|)[n]][r] (up) or U_c (down).
template <int P>
__device__ double class_entry(const double* __restrict__ W, int kpad, const uint16_t* __restrict__ pv, int k, int m, int r) {
    using K = Cls<P>;
    const int sx = K::side(k, 0), sy = K::side(k, 1), sz = K::side(k, 2);
    if (m >= sx * sy * sz) return 0.;
    const int h[3] = {m % sx, (m / sx) % sy, m / (sx * sy)};
    double s = 0.;
    int images = 0;
    for (int f = 0; f < 8; ++f) {
        int n[3];
        bool mid = false;
        for (int a = 0; a < 3; ++a) {
            const bool flip = (f >> a) & 1;
            mid |= flip && h[a] == P - 1 - h[a];
            n[a] = flip ? P - 1 - h[a] : h[a];
        }
        if (mid) continue;
        ++images;
        const double v = W[static_cast<int64_t>(pv[(n[2] * P + n[1]) * P + n[0]]) * kpad + r];
        s += __popc(k & f) & 1 ? -v : v;
    }
    return s / images;
}

// One workgroup per (row block, wave's class); grid (row blocks, 8, 2: up, down).
template <int P>
__global__ __launch_bounds__(256) void k_m2l_pack(const RowInfo* __restrict__ rows, const TauInfo* __restrict__ tau,
                                                 const uint32_t* __restrict__ pidx, const uint16_t* __restrict__ pvec,
                                                 const int32_t* __restrict__ rank, const int64_t* __restrict__ opoff,
                                                 const double* __restrict__ ops, int LD, double* __restrict__ up,
                                                 double* __restrict__ down) {
    using K = Cls<P>;
    constexpr int NN = P * P * P;
    const int rb = blockIdx.x, w = blockIdx.y;
    const bool is_up = blockIdx.z == 0;
    const int k = class_of(w), o = odd_axes(k);
    const int count = is_up ? 128 * K::ksp(o) : 256 * K::nt(o);
    double* dst = is_up ? up + static_cast<int64_t>(rb) * K::up_off(8) + K::up_off(w)
                        : down + static_cast<int64_t>(rb) * K::down_off(8) + K::down_off(w);
    for (int e = threadIdx.x; e < count; e += blockDim.x) {
        // fragments in pairs of K steps: [pair][lane][2]
        const int lane = (e / 2) % 64, pair = e / 128;
        const int i = lane & 15, kq = lane >> 4;
        int m, row;
        if (is_up) {  // K step s = 2 pair + (e & 1) over half-nodes; matrix row i is row 4 (i % 4) + i / 4
            m = 4 * (2 * pair + (e & 1)) + kq;
            row = 16 * rb + 4 * (i & 3) + (i >> 2);
        } else {  // row tile pair / 2 of half-nodes, K step s over rows 4 kq + s
            m = 16 * (pair / 2) + i;
            row = 16 * rb + 4 * kq + 2 * (pair & 1) + (e & 1);
        }
        const int t = rows[row].tau;
        double v = 0.;
        if (t != kTauDummy) {
            const TauInfo ti = tau[t];
            const int r = row - ti.row0;
            if (r < ti.rank) {
                const uint32_t ci = pidx[ti.pos];
                const int kpad = (rank[ci] + 15) & ~15;
                const double* U = ops + opoff[ci];
                v = class_entry<P>(is_up ? U + static_cast<int64_t>(NN + 1) * kpad : U, kpad,
                                   pvec + static_cast<int64_t>(ti.pos) * LD, k, m, r);
            }
        }
        dst[e] = v;
    }
}

// The tables and fragments in one device buffer: `tables` (rows, offsets, slot
// table), then the fragments of the upward and of the downward product.
template <int P>
int pack_impl(Context* c, int nrb, const std::vector<char>& tables, size_t tau_at) {
    using K = Cls<P>;
    const size_t up_at = (tables.size() + 255) & ~size_t(255);
    const size_t up = static_cast<size_t>(nrb) * K::up_off(8), down = static_cast<size_t>(nrb) * K::down_off(8);
    HFMM_TRY(ensure(c, c->d_m2lops, up_at + sizeof(double) * (up + down)));
    char* base = c->d_m2lops.as<char>();
    c->m2l_up = reinterpret_cast<double*>(base + up_at);
    c->m2l_down = c->m2l_up + up;
    HFMM_HIP(c, hipMemcpy(base, tables.data(), tables.size(), hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_m2l_pack<P>, dim3(nrb, kMWaves, 2), dim3(256), 0, c->stream,
                       reinterpret_cast<const RowInfo*>(base), reinterpret_cast<const TauInfo*>(base + tau_at),
                       c->d_pidx.as<uint32_t>(), c->d_pvec.as<uint16_t>(), c->d_rank.as<int32_t>(),
                       c->d_opoff.as<int64_t>(), c->d_ops.as<double>(), c->LD, c->m2l_up, c->m2l_down);
    return check_launch(c, "m2l_pack");
}

// Device memory for C: all of it, or what kRoomMax and workspace_room leave.
// Beyond that the rows run in parts, each with the prologue of every tile and
// with partial locals through memory (p^3 doubles per cell and part).  Within a
// buffer's reach (4 GB) the upward kernel stores through a buffer; beyond it
// with 64-bit addresses under a mask, which costs less than the parts: 1M uniform
// h7, order 7 (12 GB) 17.2 ms in three parts, 16.4 in one; 192 sets x 8 vectors,
// order 5, 51.0 / 48.5; 12M uniform h9, order 5, a pass of 2,783 ms one step at a
// time, 730 with 32 GB, 530 with 64.
constexpr int kMaxPart = 116;  // row blocks of a launch: their table fits the LDS beside the tiles
constexpr size_t kRoomMax = size_t(32) << 30;

// Bytes of the workspaces of the process on each device.
std::atomic<size_t> g_held[64];

// Bytes that the workspace may take of `want`.  The device is asked where a tree
// wants more than before, and not again until the next build, so that a captured
// run decides as the run before it and memory that was freed since then counts.
size_t room_of(Context* c, size_t want) {
    if (want > c->m2l_asked) {
        c->m2l_asked = want;
        const size_t own = c->d_m2lC.bytes + c->d_m2lacc.bytes;
        if (c->d_m2lC.bytes >= want) {
            c->m2l_room = want;
        } else {
            size_t free_b = 0, total_b = 0;
            if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) (void)hipGetLastError();
            c->m2l_room = workspace_room(want, own, std::max(own, g_held[c->device].load()), free_b);
        }
    }
    return std::min(want, c->m2l_room);
}

// acc: bytes of the partial locals
template <int P, int C, bool WIDE>
int m2l_launch(Context* c, M2LArgs a, size_t acc, size_t room) {
    using K = Cls<P>;
    constexpr int RB = Lds<C>::RB;
    const int64_t tiles = (a.ncell + 16 * C - 1) / (16 * C);
    const int64_t grid = (tiles + 8 * kXcdChunk - 1) / (8 * kXcdChunk) * (8 * kXcdChunk);
    std::vector<int> cut;
    int parts = 0;
    for (;;) {  // where the device refuses, smaller parts
        const size_t bytes = cut_rows(c->m2l_rboff, RB, kMaxPart, a.ncell, acc, room, cut);
        parts = static_cast<int>(cut.size()) - 1;
        int st = parts > 1 ? ensure(c, c->d_m2lacc, acc) : HFMM_OK;
        if (st == HFMM_OK) st = ensure(c, c->d_m2lC, bytes);
        count_m2l_workspace(c);
        if (st == HFMM_OK) break;
        if (st != HFMM_ERR_NOMEM || parts * RB >= c->m2l_nrb) return st;
        HFMM_HIP(c, hipStreamSynchronize(c->stream));
        release(c->d_m2lC);
        c->m2l_room = room = (bytes + (parts > 1 ? acc : 0)) / 2;
    }
    a.C = c->d_m2lC.as<double>();
    a.acc = c->d_m2lacc.as<double>();
    int maxrows = 0;
    for (int i = 0; i < parts; ++i) maxrows = std::max(maxrows, 16 * (cut[i + 1] - cut[i]));
    const int tilebuf = 2 * Lds<C>::kBuf;
    const SmemLayout su = smem_layout(std::max(tilebuf, K::exp_off(8)), 16 * C * kTgtRow * 4, maxrows);
    const SmemLayout sd = smem_layout(std::max(tilebuf, 17 * K::loc_off(8)), 16 * C * kTauStride, 0);
    static int lds_up[64] = {0}, lds_down[64] = {0};
    HFMM_TRY(raise_lds_limit(c, reinterpret_cast<const void*>(&k_m2l_up<P, C, WIDE>), su.bytes, lds_up));
    HFMM_TRY(raise_lds_limit(c, reinterpret_cast<const void*>(&k_m2l_down<P, C>), sd.bytes, lds_down));
    for (int i = 0; i < parts; ++i) {
        a.rb0 = cut[i];
        a.rb1 = cut[i + 1];
        a.off0 = c->m2l_rboff[cut[i]];
        a.stride = c->m2l_rboff[cut[i + 1]] - a.off0;
        a.load = i > 0;
        a.store = i + 1 < parts;
        a.ops = c->m2l_up;
        prof_begin(c, is_mixed(c) ? "m2l_mixed" : "m2l");
        hipLaunchKernelGGL((k_m2l_up<P, C, WIDE>), dim3(static_cast<unsigned>(grid)), dim3(kMThreads), su.bytes, c->stream, a,
                           su, c->d_M.as<double>(), c->LD);
        prof_end(c);
        HFMM_TRY(check_launch(c, "m2l_up"));
        a.ops = c->m2l_down;
        prof_begin(c, is_mixed(c) ? "m2l_mixed" : "m2l");
        hipLaunchKernelGGL((k_m2l_down<P, C>), dim3(static_cast<unsigned>(grid)), dim3(kMThreads), sd.bytes, c->stream,
                           a, sd, c->d_L.as<double>(), c->LD);
        prof_end(c);
        HFMM_TRY(check_launch(c, "m2l_down"));
    }
    return HFMM_OK;
}

template <int P>
int m2l_impl(Context* c) {
    int unused = 0;
    M2LArgs a{};
    a.lv = make_levels(c, 16, unused);
    if (a.lv.nlev == 0) return HFMM_OK;  // no M2L level in the working range
    const int last = a.lv.pcount_off[a.lv.nlev - 1] / 8;
    a.first = a.lv.cell_off[0];
    a.ncell = a.lv.cell_off[a.lv.nlev - 1] + c->ncell[last] - a.first;
    if (a.ncell <= 0) return HFMM_OK;
    a.slots = c->d_m2l.as<int32_t>();
    a.keys = c->d_cellkey.as<uint64_t>();
    a.rows = c->d_m2lops.as<RowInfo>();
    a.slot_tau = reinterpret_cast<const uint16_t*>(c->d_m2lops.as<char>() + c->m2l_slots_at);
    int step = 0;
    for (int b = 0; b < c->m2l_nrb; ++b) step = std::max(step, c->m2l_rboff[b + 1] - c->m2l_rboff[b]);
    const size_t all = static_cast<size_t>(c->m2l_rboff[c->m2l_nrb]) * a.ncell;
    const size_t acc = sizeof(double) * 256 * Cls<P>::nt(0) * kMWaves * 2 * static_cast<size_t>((a.ncell + 31) / 32);
    const bool parts = all > kRoomMax || c->m2l_nrb > kMaxPart;
    const size_t room = room_of(c, std::min(all, kRoomMax) + (parts ? acc : 0));
    if (room > kBufferMax || static_cast<size_t>(step) * a.ncell > kBufferMax) return m2l_launch<P, 2, true>(c, a, acc, room);
    return two_tiles(a.ncell) ? m2l_launch<P, 2, false>(c, a, acc, room) : m2l_launch<P, 1, false>(c, a, acc, room);
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

// Tables and operator fragments of the uploaded symmetric operators.
int prepare_m2l_f64(Context* c) {
    const ChebOperators& op = c->ops;
    TauInfo tau[kTau];
    int tau_of[4][4][4];
    int n = 0, row = 0;
    for (int x = 0; x < 4; ++x)
        for (int y = 0; y < 4; ++y)
            for (int z = 0; z < 4; ++z) {
                tau_of[x][y][z] = -1;
                if (x < 2 && y < 2 && z < 2) continue;
                TauInfo& t = tau[n];
                t.pos = ((x + 3) * 7 + y + 3) * 7 + z + 3;
                t.rank = op.rank[op.pidx[t.pos]];
                t.row0 = row;
                t.pad = 0;
                row += (t.rank + 3) & ~3;
                tau_of[x][y][z] = n++;
            }
    const int nrb = ((row + 15) / 16 + 1) & ~1;  // whole steps of either tile shape
    if (n != kTau || nrb > kMaxSteps) return fail(c, HFMM_ERR_ARG, "operator rank above 64 is not supported");
    std::vector<uint16_t> slot_tau(2 * 8 * kFarSlots);
    for (int e = 0; e < 8; ++e) {
        FarSlot fs[kFarSlots];
        far_slots(e, fs);
        for (int j = 0; j < kFarSlots; ++j) {
            const int d[3] = {fs[j].pos / 49 - 3, (fs[j].pos / 7) % 7 - 3, fs[j].pos % 7 - 3};
            const int t = tau_of[std::abs(d[0])][std::abs(d[1])][std::abs(d[2])];
            int s = 0, back = 0;  // signs of the slot's position, and of the position seen from the other cell
            for (int a = 0; a < 3; ++a) {
                if (d[a] < 0) s |= 1 << a;
                if (d[a] > 0) back |= 1 << a;
            }
            slot_tau[e * kFarSlots + j] = static_cast<uint16_t>(8 * t + s);
            slot_tau[(8 + e) * kFarSlots + j] = static_cast<uint16_t>(8 * t + back);
        }
    }
    std::vector<RowInfo> rows;
    row_layout(tau, nrb, rows, c->m2l_rboff);
    const size_t tau_at = sizeof(RowInfo) * rows.size();
    c->m2l_slots_at = tau_at + sizeof(tau);
    std::vector<char> tables(c->m2l_slots_at + sizeof(uint16_t) * slot_tau.size());
    std::memcpy(tables.data(), rows.data(), tau_at);
    std::memcpy(tables.data() + tau_at, tau, sizeof(tau));
    std::memcpy(tables.data() + c->m2l_slots_at, slot_tau.data(), sizeof(uint16_t) * slot_tau.size());
    // an earlier evaluation may still read the old tables
    HFMM_HIP(c, hipStreamSynchronize(c->stream));
    const auto pack = [&] {
#define CALL(P) pack_impl<P>(c, nrb, tables, tau_at)
        HFMM_DISPATCH(c->order(), CALL)
#undef CALL
    };
    HFMM_TRY(pack());
    c->m2l_nrb = nrb;  // prepared: not before the memory is there and the kernel on its way
    return HFMM_OK;
}

void count_m2l_workspace(Context* c) {
    const size_t now = c->d_m2lC.bytes + c->d_m2lacc.bytes;
    if (now == c->m2l_counted) return;
    g_held[c->device] += now - c->m2l_counted;  // modulo 2^64
    c->m2l_counted = now;
}

int run_m2l(Context* c) {
#define CALL(P) m2l_impl<P>(c)
    HFMM_DISPATCH(c->order(), CALL)
#undef CALL
}

}  // namespace hfmm

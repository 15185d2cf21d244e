// tree_device.hip -- octree construction on the device (FP64 keys, int32
// indices): leaf coordinates and Morton keys, a stable LSD radix sort,
// run-length encoded leaves, parent levels, P2P neighbour slots and M2L
// interaction slots in the reference's enumeration order.
//
// Follows (reference paths relative to its source tree):
//   coordinates   Src/Containers/FCoordinateComputer.hpp:15-24, 42-54
//   Morton keys   Src/Containers/FTreeCoordinate.hpp:91-142
//   sort/leaves   Src/GroupTree/Core/FGroupTree.hpp:192-360
//   P2P list      Src/Containers/FTreeCoordinate.hpp:189-214
//   M2L list      Src/Containers/FTreeCoordinate.hpp:219-264
#include <hip/hip_runtime.h>

#include <algorithm>

#include "hfmm_internal.hpp"

namespace hfmm {
namespace {

constexpr int kBlock = 256;
constexpr int kItems = 8;
constexpr int kTile = kBlock * kItems;  // elements per scan / sort tile

// ---------------------------------------------------------------------------
// Morton helpers: bit 3k <- z_k, 3k+1 <- y_k, 3k+2 <- x_k.
__device__ __forceinline__ uint64_t spread3(uint32_t v) {
    uint64_t x = v & 0x1fffffu;
    x = (x | (x << 32)) & 0x1f00000000ffffull;
    x = (x | (x << 16)) & 0x1f0000ff0000ffull;
    x = (x | (x << 8)) & 0x100f00f00f00f00full;
    x = (x | (x << 4)) & 0x10c30c30c30c30c3ull;
    x = (x | (x << 2)) & 0x1249249249249249ull;
    return x;
}
__device__ __forceinline__ uint32_t compact3(uint64_t x) {
    x &= 0x1249249249249249ull;
    x = (x ^ (x >> 2)) & 0x10c30c30c30c30c3ull;
    x = (x ^ (x >> 4)) & 0x100f00f00f00f00full;
    x = (x ^ (x >> 8)) & 0x1f0000ff0000ffull;
    x = (x ^ (x >> 16)) & 0x1f00000000ffffull;
    x = (x ^ (x >> 32)) & 0x1fffffull;
    return static_cast<uint32_t>(x);
}
__device__ __forceinline__ uint64_t morton3(int x, int y, int z) {
    return (spread3(x) << 2) | (spread3(y) << 1) | spread3(z);
}
__device__ __forceinline__ void demorton3(uint64_t k, int& x, int& y, int& z) {
    z = compact3(k);
    y = compact3(k >> 1);
    x = compact3(k >> 2);
}

// Index of a key among the sorted keys of one level (-1 when absent): a
// dense Morton -> index table when the level is small enough, otherwise a
// lower-bound search.
struct KeyIndex {
    const uint64_t* keys;
    int n;
    const int32_t* dense;  // 8^level entries or null
    __device__ __forceinline__ int find(uint64_t key) const {
        if (dense) return dense[key];
        int lo = 0, hi = n;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (keys[mid] < key) lo = mid + 1; else hi = mid;
        }
        return (lo < n && keys[lo] == key) ? lo : -1;
    }
};

// ---------------------------------------------------------------------------
// Exclusive scan (three passes: tile sums, scan of tile sums, tile scans).
template <typename T>
__device__ T block_exclusive_scan(T v, T* sh, T& total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    T incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const T add = __shfl_up(incl, d);
        if (lane >= d) incl += add;
    }
    if (lane == 63) sh[wave] = incl;
    __syncthreads();
    T before = 0, sum = 0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) {
        if (w < wave) before += sh[w];
        sum += sh[w];
    }
    __syncthreads();  // sh may be written again
    total = sum;
    return before + incl - v;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_scan_reduce(const T* __restrict__ in, int64_t n, T* __restrict__ part) {
    __shared__ T sh[kBlock];
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kTile + threadIdx.x * kItems;
    T s = 0;
    for (int i = 0; i < kItems; ++i)
        if (base + i < n) s += in[base + i];
    T total;
    block_exclusive_scan<T>(s, sh, total);
    if (threadIdx.x == 0) part[blockIdx.x] = total;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_scan_top(T* __restrict__ part, int64_t nparts, T* __restrict__ total_out) {
    __shared__ T sh[kBlock];
    T carry = 0;
    for (int64_t c0 = 0; c0 < nparts; c0 += kTile) {
        const int64_t base = c0 + threadIdx.x * kItems;
        T v[kItems];
        T s = 0;
        for (int i = 0; i < kItems; ++i) {
            v[i] = base + i < nparts ? part[base + i] : T(0);
            s += v[i];
        }
        T tot;
        T ex = block_exclusive_scan<T>(s, sh, tot) + carry;
        for (int i = 0; i < kItems; ++i) {
            if (base + i < nparts) part[base + i] = ex;
            ex += v[i];
        }
        carry += tot;
    }
    if (threadIdx.x == 0 && total_out) *total_out = carry;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_scan_apply(const T* in, T* out, int64_t n, const T* __restrict__ part) {
    __shared__ T sh[kBlock];
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kTile + threadIdx.x * kItems;
    T v[kItems];
    T s = 0;
    for (int i = 0; i < kItems; ++i) {
        v[i] = base + i < n ? in[base + i] : T(0);
        s += v[i];
    }
    T tot;
    T ex = block_exclusive_scan<T>(s, sh, tot) + part[blockIdx.x];
    for (int i = 0; i < kItems; ++i) {
        if (base + i < n) out[base + i] = ex;
        ex += v[i];
    }
}

// The whole scan by one workgroup: for few tiles the launches of the other
// kernels cost more than the loop over them (about 2 us each).
constexpr int64_t kScanOneTiles = 8;

template <typename T>
__global__ __launch_bounds__(kBlock) void k_scan_one(const T* in, T* out, int64_t n, T* __restrict__ total_out) {
    __shared__ T sh[kBlock];
    T carry = 0;
    for (int64_t c0 = 0; c0 < n; c0 += kTile) {
        const int64_t base = c0 + threadIdx.x * kItems;
        T v[kItems];
        T s = 0;
        for (int i = 0; i < kItems; ++i) {
            v[i] = base + i < n ? in[base + i] : T(0);
            s += v[i];
        }
        T tot;
        T ex = block_exclusive_scan<T>(s, sh, tot) + carry;
        for (int i = 0; i < kItems; ++i) {
            if (base + i < n) out[base + i] = ex;
            ex += v[i];
        }
        carry += tot;
    }
    if (threadIdx.x == 0) *total_out = carry;
}

// out = exclusive scan of in (may alias); *total_dev = sum.
template <typename T>
int exclusive_scan(Context* c, const T* in, T* out, int64_t n, T* total_dev, const char* tag) {
    if (n <= 0) {
        HFMM_HIP(c, hipMemsetAsync(total_dev, 0, sizeof(T), c->stream));
        return HFMM_OK;
    }
    const int64_t tiles = (n + kTile - 1) / kTile;
    if (tiles <= kScanOneTiles) {
        prof_begin(c, tag);
        hipLaunchKernelGGL(k_scan_one<T>, dim3(1), dim3(kBlock), 0, c->stream, in, out, n, total_dev);
        prof_end(c);
        return check_launch(c, tag);
    }
    HFMM_TRY(ensure(c, c->d_scan_part, sizeof(T) * static_cast<size_t>(tiles + 1)));
    T* part = c->d_scan_part.as<T>();
    prof_begin(c, tag);
    hipLaunchKernelGGL(k_scan_reduce<T>, dim3(static_cast<unsigned>(tiles)), dim3(kBlock), 0, c->stream, in, n, part);
    hipLaunchKernelGGL(k_scan_top<T>, dim3(1), dim3(kBlock), 0, c->stream, part, tiles, total_dev);
    hipLaunchKernelGGL(k_scan_apply<T>, dim3(static_cast<unsigned>(tiles)), dim3(kBlock), 0, c->stream, in, out, n,
                       part);
    prof_end(c);
    return check_launch(c, tag);
}

// ---------------------------------------------------------------------------
// Stable LSD radix sort of (uint64 key, int32 value), 8-bit digits.
__global__ __launch_bounds__(kBlock) void k_radix_hist(const uint64_t* __restrict__ keys, int64_t n, int shift,
                                                      int32_t* __restrict__ hist, int64_t ntiles) {
    __shared__ int32_t s[256];
    s[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kTile;
    for (int r = 0; r < kItems; ++r) {
        const int64_t e = base + r * kBlock + threadIdx.x;
        if (e < n) atomicAdd(&s[(keys[e] >> shift) & 255u], 1);
    }
    __syncthreads();
    hist[static_cast<int64_t>(threadIdx.x) * ntiles + blockIdx.x] = s[threadIdx.x];
}

// Scatter one tile: elements are visited in rounds of 256 consecutive
// elements; within a wave the rank among equal digits comes from ballots,
// across the four waves from per-digit counters, so the order of equal keys
// is preserved.
__global__ __launch_bounds__(kBlock) void k_radix_scatter(const uint64_t* __restrict__ kin,
                                                         const int32_t* __restrict__ vin, int64_t n, int shift,
                                                         const int32_t* __restrict__ offs, int64_t ntiles,
                                                         uint64_t* __restrict__ kout, int32_t* __restrict__ vout) {
    __shared__ int32_t s_base[256];
    __shared__ int32_t s_wave[4][256];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    s_base[tid] = offs[static_cast<int64_t>(tid) * ntiles + blockIdx.x];
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kTile;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int r = 0; r < kItems; ++r) {
        const int64_t e = base + r * kBlock + tid;
        const bool valid = e < n;
        const uint64_t key = valid ? kin[e] : 0ull;
        const int digit = valid ? static_cast<int>((key >> shift) & 255u) : 0;
        for (int w = 0; w < 4; ++w) s_wave[w][tid] = 0;
        __syncthreads();
        uint64_t peers = __ballot(valid);
        for (int b = 0; b < 8; ++b) {
            const bool bit = (digit >> b) & 1;
            const uint64_t m = __ballot(bit);
            peers &= bit ? m : ~m;
        }
        const int rank = __popcll(peers & lt_mask);
        if (valid && rank == 0) s_wave[wave][digit] = __popcll(peers);
        __syncthreads();
        {
            int run = s_base[tid];
            for (int w = 0; w < 4; ++w) {
                const int cnt = s_wave[w][tid];
                s_wave[w][tid] = run;
                run += cnt;
            }
            s_base[tid] = run;
        }
        __syncthreads();
        if (valid) {
            const int dst = s_wave[wave][digit] + rank;
            kout[dst] = key;
            vout[dst] = vin[e];
        }
        __syncthreads();
    }
}

// Sorts (keys, vals) by the low `nbits` bits of the keys, using the second
// buffers; `swapped`: the result ends in keys2 / vals2.
int radix_sort(Context* c, uint64_t* keys, int32_t* vals, uint64_t* keys2, int32_t* vals2, int64_t n, int nbits,
               bool& swapped) {
    swapped = false;
    if (n <= 1) return HFMM_OK;
    const int64_t ntiles = (n + kTile - 1) / kTile;
    HFMM_TRY(ensure(c, c->d_hist, sizeof(int32_t) * static_cast<size_t>(256 * ntiles + 1)));
    HFMM_TRY(ensure(c, c->d_count, sizeof(int64_t) * 24));
    int32_t* hist = c->d_hist.as<int32_t>();
    const int passes = (nbits + 7) / 8;
    uint64_t *ka = keys, *kb = keys2;
    int32_t *va = vals, *vb = vals2;
    for (int p = 0; p < passes; ++p) {
        prof_begin(c, "radix_hist");
        hipLaunchKernelGGL(k_radix_hist, dim3(static_cast<unsigned>(ntiles)), dim3(kBlock), 0, c->stream, ka, n, 8 * p,
                           hist, ntiles);
        prof_end(c);
        HFMM_TRY(check_launch(c, "radix_hist"));
        HFMM_TRY(exclusive_scan<int32_t>(c, hist, hist, 256 * ntiles,
                                         reinterpret_cast<int32_t*>(c->d_count.as<int64_t>() + 15), "radix_scan"));
        prof_begin(c, "radix_scatter");
        hipLaunchKernelGGL(k_radix_scatter, dim3(static_cast<unsigned>(ntiles)), dim3(kBlock), 0, c->stream, ka, va, n,
                           8 * p, hist, ntiles, kb, vb);
        prof_end(c);
        HFMM_TRY(check_launch(c, "radix_scatter"));
        std::swap(ka, kb);
        std::swap(va, vb);
    }
    swapped = ka != keys;
    return HFMM_OK;
}

// ---------------------------------------------------------------------------
// Leaf coordinates and keys (FCoordinateComputer::GetTreeCoordinate):
// c = rel == width ? 2^(h-1)-1 : int(rel / leafwidth), rel in [0, width].
// With particle sets the key is (set << 3(h-1)) | set-local key; the set of a
// particle is found by bisection of the set offsets.
__global__ __launch_bounds__(kBlock) void k_morton(int64_t n, const double* __restrict__ x,
                                                  const double* __restrict__ y, const double* __restrict__ z,
                                                  double cx, double cy, double cz, double width, double leafw,
                                                  int lbits, const int64_t* __restrict__ setoff, int nsets,
                                                  uint64_t* __restrict__ keys, int32_t* __restrict__ vals,
                                                  int32_t* __restrict__ err) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int lim = 1 << lbits;
    const double rel[3] = {x[i] - cx, y[i] - cy, z[i] - cz};
    int co[3];
    bool bad = false;
    for (int d = 0; d < 3; ++d) {
        if (!(rel[d] >= 0 && rel[d] <= width)) { bad = true; co[d] = 0; continue; }
        co[d] = rel[d] == width ? lim - 1 : static_cast<int>(rel[d] / leafw);
        if (co[d] >= lim) { bad = true; co[d] = lim - 1; }
    }
    if (bad) atomicOr(err, 1);
    uint64_t set = 0;
    if (setoff) {  // last set whose first particle is <= i
        int lo = 0, hi = nsets - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (setoff[mid] <= i) lo = mid; else hi = mid - 1;
        }
        set = static_cast<uint64_t>(lo);
    }
    keys[i] = (set << (3 * lbits)) | morton3(co[0], co[1], co[2]);
    vals[i] = static_cast<int32_t>(i);
}

// The sorted particles, and the inverse of the sort permutation (input index ->
// sorted index), through which the results go back to the input order.
__global__ __launch_bounds__(kBlock) void k_gather_particles(int64_t n, const int32_t* __restrict__ idx,
                                                            const double* __restrict__ x, const double* __restrict__ y,
                                                            const double* __restrict__ z, const double* __restrict__ q,
                                                            double* __restrict__ out, int32_t* __restrict__ iperm) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    // the padding that masked sources read: their charge has to be a number
    if (i == 0)
        for (int k = 0; k < kSortedPad; ++k) out[4 * n + k] = 0.;
    const int32_t o = idx[i];
    iperm[o] = static_cast<int32_t>(i);
    out[i] = x[o];
    out[n + i] = y[o];
    out[2 * n + i] = z[o];
    out[3 * n + i] = q[o];
}

// New charges on an existing tree: sorted q[i] = q_in[perm[i]].
__global__ __launch_bounds__(kBlock) void k_gather_charges(int64_t n, const int32_t* __restrict__ perm,
                                                          const double* __restrict__ q, double* __restrict__ sq) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    sq[i] = q[perm[i]];
}

// The sorted charges of vectors r0 .. r0 + R - 1 as [n][R] (T = float: the
// mixed forms' P2P charges, rounded as k_local_coords rounds them).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_gather_charge_chunk(int64_t n, const int32_t* __restrict__ perm,
                                                               const double* __restrict__ q, int r0, int R,
                                                               T* __restrict__ out) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t o = perm[i];
    for (int r = 0; r < R; ++r) out[i * R + r] = static_cast<T>(q[static_cast<int64_t>(r0 + r) * n + o]);
}

// The cells of every level from the sorted particle keys at once: particle i
// begins a cell of level l where its key differs from the one before it in the
// bits above the levels below l.  k_level_counts counts the cells per tile and
// level (and the leaves of more than kP2PBig particles: key i + kP2PBig is the
// same), k_level_scan scans the tiles of each level, k_level_cells writes.  Level
// by level (flags, scan, write, the count to the host) a tree of height 5 took 24
// launches and 4 waits.
struct TreeLevels {
    int top, leaf;                    // first and last level
    int64_t lvl_off[kMaxLevels + 1];  // cells before each level
    int64_t cs_off[kMaxLevels];       // child ranges of each level
    int64_t ncell[kMaxLevels];
};

// The highest level at which i begins a cell (leaf + 1: none).
__device__ __forceinline__ int head_level(uint64_t key, uint64_t before, int64_t i, int top, int leaf) {
    if (i == 0) return top;
    const uint64_t d = key ^ before;
    if (d == 0) return leaf + 1;
    return max(top, leaf - (63 - __clzll(d)) / 3);
}

__global__ __launch_bounds__(kBlock) void k_level_counts(int64_t n, const uint64_t* __restrict__ keys, int top, int leaf,
                                                        int64_t ntiles, int32_t* __restrict__ counts,
                                                        int32_t* __restrict__ nbig) {
    __shared__ int32_t s[kMaxLevels + 1];
    if (threadIdx.x <= kMaxLevels) s[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kTile;
    int big = 0;
    for (int r = 0; r < kItems; ++r) {
        const int64_t i = base + r * kBlock + threadIdx.x;
        if (i >= n) break;
        const uint64_t key = keys[i];
        const int h = head_level(key, i ? keys[i - 1] : 0ull, i, top, leaf);
        if (h > leaf) continue;
        atomicAdd(&s[h], 1);
        if (i + kP2PBig < n && keys[i + kP2PBig] == key) ++big;
    }
    if (big) atomicAdd(nbig, big);
    __syncthreads();
    if (threadIdx.x == 0) {
        int sum = 0;  // a cell that begins at level h begins one at every level below
        for (int l = top; l <= leaf; ++l) {
            sum += s[l];
            counts[static_cast<int64_t>(l - top) * ntiles + blockIdx.x] = sum;
        }
    }
}

// One workgroup per level: exclusive scan of its tiles, the sum to total[level].
__global__ __launch_bounds__(kBlock) void k_level_scan(int64_t ntiles, int32_t* __restrict__ counts,
                                                      int32_t* __restrict__ total) {
    __shared__ int32_t sh[kBlock];
    int32_t* c = counts + static_cast<int64_t>(blockIdx.x) * ntiles;
    int32_t carry = 0;
    for (int64_t c0 = 0; c0 < ntiles; c0 += kTile) {
        const int64_t base = c0 + threadIdx.x * kItems;
        int32_t v[kItems], sum = 0;
        for (int i = 0; i < kItems; ++i) {
            v[i] = base + i < ntiles ? c[base + i] : 0;
            sum += v[i];
        }
        int32_t tot;
        int32_t ex = block_exclusive_scan<int32_t>(sum, sh, tot) + carry;
        for (int i = 0; i < kItems; ++i) {
            if (base + i < ntiles) c[base + i] = ex;
            ex += v[i];
        }
        carry += tot;
    }
    if (threadIdx.x == 0) total[blockIdx.x] = carry;
}

__global__ __launch_bounds__(kBlock) void k_level_cells(int64_t n, const uint64_t* __restrict__ keys, TreeLevels lv,
                                                       int64_t ntiles, const int32_t* __restrict__ counts,
                                                       uint64_t* __restrict__ cellkey, int32_t* __restrict__ cstart,
                                                       int32_t* __restrict__ lstart, int32_t* __restrict__ pleaf) {
    __shared__ int32_t sh[kBlock];
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kTile + threadIdx.x * kItems;
    uint64_t key[kItems];
    int head[kItems];
    for (int i = 0; i < kItems; ++i) {
        key[i] = 0;
        head[i] = lv.leaf + 1;
        if (base + i >= n) continue;
        key[i] = keys[base + i];
        const uint64_t before = i ? key[i - 1] : base ? keys[base - 1] : 0ull;
        head[i] = head_level(key[i], before, base + i, lv.top, lv.leaf);
    }
    int32_t below[kItems];  // index of each particle's cell in the level below
    for (int l = lv.leaf; l >= lv.top; --l) {
        int32_t sum = 0;
        for (int i = 0; i < kItems; ++i) sum += head[i] <= l;
        int32_t tot;
        int32_t at = block_exclusive_scan<int32_t>(sum, sh, tot) +
                     counts[static_cast<int64_t>(l - lv.top) * ntiles + blockIdx.x] - 1;
        for (int i = 0; i < kItems; ++i) {
            if (base + i >= n) break;
            if (head[i] <= l) {
                ++at;
                cellkey[lv.lvl_off[l] + at] = key[i] >> (3 * (lv.leaf - l));
                if (l == lv.leaf) lstart[at] = static_cast<int32_t>(base + i);
                else cstart[lv.cs_off[l] + at] = below[i];
            }
            if (l == lv.leaf) pleaf[base + i] = at;
            below[i] = at;
        }
    }
    // the ends of the ranges
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        lstart[lv.ncell[lv.leaf]] = static_cast<int32_t>(n);
        for (int l = lv.leaf - 1; l >= lv.top; --l)
            cstart[lv.cs_off[l] + lv.ncell[l]] = static_cast<int32_t>(lv.ncell[l + 1]);
    }
}

// The levels of a launch over cells: level i owns workgroups first[i] ..
// first[i + 1] - 1, kSlotCells cells each.
constexpr int kSlotCells = 32;
struct SlotLevels {
    int nlev;
    int first[kMaxLevels + 1];
    KeyIndex ix[kMaxLevels];
    int lim[kMaxLevels];  // cells per axis of one set
    int64_t cell_off[kMaxLevels];
};

// Morton -> cell tables of the levels that have one.
__global__ __launch_bounds__(kBlock) void k_dense_index(SlotLevels lv) {
    const int bid = blockIdx.x;
    if (bid >= lv.first[lv.nlev]) return;
    int li = 0;
    while (bid >= lv.first[li + 1]) ++li;
    const int i = (bid - lv.first[li]) * kSlotCells + threadIdx.x;
    if (static_cast<int>(threadIdx.x) < kSlotCells && i < lv.ix[li].n && lv.ix[li].dense)
        const_cast<int32_t*>(lv.ix[li].dense)[lv.ix[li].keys[i]] = i;
}

// Slots of every cell of the launch's levels, one entry per thread and turn: the
// cell at a given offset of each slot (the key by dilated additions on the
// cell's own, which is decoded once), or -1 where it is empty or outside the set's
// box.  P2P: the 26 neighbours in position order; M2L: the 189 slots of the cell's
// parity in the reference enumeration order (offset -> position, slotpos).  A cell
// at such an offset has its parent beside the cell's, so the box test on the cell
// is that of the parents.  One thread per cell wrote its slots one by one, 104
// or 756 bytes from its neighbour's: 163 us for the 262,144 leaves of a 1M tree.
template <int NSLOT, bool FAR>
__global__ __launch_bounds__(kBlock) void k_cell_slots(SlotLevels lv, const int16_t* __restrict__ slotpos,
                                                      int32_t* __restrict__ slots) {
    constexpr uint64_t MX = 0x4924924924924924ull, MY = 0x2492492492492492ull, MZ = 0x1249249249249249ull;
    __shared__ uint64_t s_key[kSlotCells];
    __shared__ int s_pos[kSlotCells][4];  // set-local coordinates, parity
    __shared__ int16_t s_off[FAR ? 8 * NSLOT : 1];
    __shared__ uint64_t s_dil[7];
    const int bid = blockIdx.x;
    if (bid >= lv.first[lv.nlev]) return;
    int li = 0;
    while (bid >= lv.first[li + 1]) ++li;
    const KeyIndex ix = lv.ix[li];
    const int lim = lv.lim[li];
    const int cell0 = (bid - lv.first[li]) * kSlotCells;
    const int cnt = min(kSlotCells, ix.n - cell0);
    if (static_cast<int>(threadIdx.x) < cnt) {
        const uint64_t key = ix.keys[cell0 + threadIdx.x];
        int x, y, z;
        demorton3(key, x, y, z);
        s_key[threadIdx.x] = key;
        s_pos[threadIdx.x][0] = x & (lim - 1);
        s_pos[threadIdx.x][1] = y & (lim - 1);
        s_pos[threadIdx.x][2] = z & (lim - 1);
        s_pos[threadIdx.x][3] = static_cast<int>(key & 7u);
    }
    if (threadIdx.x < 7) s_dil[threadIdx.x] = spread3(static_cast<uint32_t>(static_cast<int>(threadIdx.x) - 3) & 0x1fffffu);
    if (FAR)
        for (int i = threadIdx.x; i < 8 * NSLOT; i += kBlock) s_off[i] = slotpos[i];
    __syncthreads();
    int32_t* out = slots + (lv.cell_off[li] + cell0) * NSLOT;
    for (int e = threadIdx.x; e < cnt * NSLOT; e += kBlock) {
        const int c = e / NSLOT, j = e - c * NSLOT;
        int dx, dy, dz;
        if (FAR) {
            const int pos = s_off[s_pos[c][3] * NSLOT + j];
            dx = pos / 49 - 3, dy = (pos / 7) % 7 - 3, dz = pos % 7 - 3;
        } else {
            const int pos = j < 13 ? j : j + 1;
            dx = pos / 9 - 1, dy = (pos / 3) % 3 - 1, dz = pos % 3 - 1;
        }
        const int nx = s_pos[c][0] + dx, ny = s_pos[c][1] + dy, nz = s_pos[c][2] + dz;
        int f = -1;
        if (nx >= 0 && nx < lim && ny >= 0 && ny < lim && nz >= 0 && nz < lim) {
            const uint64_t key = s_key[c];
            const uint64_t kx = ((key | ~MX) + (s_dil[dx + 3] << 2)) & MX;
            const uint64_t ky = ((key | ~MY) + (s_dil[dy + 3] << 1)) & MY;
            const uint64_t kz = ((key | ~MZ) + s_dil[dz + 3]) & MZ;
            f = ix.find(kx | ky | kz);
        }
        out[e] = f;
    }
}

// Cells of a level grouped by child index (stable), every level in one launch:
// per tile of kTile cells the counts of the 8 parities, their scan over the
// tiles of the level, parity by parity, and the places.  Eight 16-bit counters
// in two words.
struct ParityLevels {
    int nlev;
    int first[kMaxLevels + 1];  // tiles before each level
    int64_t cell_off[kMaxLevels];
    int ncell[kMaxLevels];
    int level[kMaxLevels];
};

__global__ __launch_bounds__(kBlock) void k_parity_counts(ParityLevels lv, const uint64_t* __restrict__ cellkey,
                                                         int32_t* __restrict__ counts) {
    __shared__ int32_t s[8];
    int li = 0;
    while (static_cast<int>(blockIdx.x) >= lv.first[li + 1]) ++li;
    if (threadIdx.x < 8) s[threadIdx.x] = 0;
    __syncthreads();
    const int base = (static_cast<int>(blockIdx.x) - lv.first[li]) * kTile;
    for (int r = 0; r < kItems; ++r) {
        const int i = base + r * kBlock + static_cast<int>(threadIdx.x);
        if (i < lv.ncell[li]) atomicAdd(&s[cellkey[lv.cell_off[li] + i] & 7u], 1);
    }
    __syncthreads();
    if (threadIdx.x < 8) counts[blockIdx.x * 8 + threadIdx.x] = s[threadIdx.x];
}

// One workgroup per level: counts[tile][parity] -> first place of the tile's
// cells of that parity; pcount[level][parity].
__global__ __launch_bounds__(64) void k_parity_scan(ParityLevels lv, int32_t* __restrict__ counts,
                                                   int32_t* __restrict__ pcount) {
    __shared__ int32_t s_sum[8], s_start[8];
    const int li = blockIdx.x, lane = threadIdx.x;
    const int t0 = lv.first[li], t1 = lv.first[li + 1];
    if (lane < 8) {
        int sum = 0;
        for (int t = t0; t < t1; ++t) sum += counts[t * 8 + lane];
        s_sum[lane] = sum;
        pcount[8 * lv.level[li] + lane] = sum;
    }
    __syncthreads();
    if (lane == 0) {
        int run = 0;
        for (int p = 0; p < 8; ++p) {
            s_start[p] = run;
            run += s_sum[p];
        }
    }
    __syncthreads();
    if (lane < 8) {
        int run = s_start[lane];
        for (int t = t0; t < t1; ++t) {
            const int c = counts[t * 8 + lane];
            counts[t * 8 + lane] = run;
            run += c;
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_parity_order(ParityLevels lv, const uint64_t* __restrict__ cellkey,
                                                        const int32_t* __restrict__ counts, int32_t* __restrict__ order) {
    __shared__ uint64_t sh[kBlock];
    int li = 0;
    while (static_cast<int>(blockIdx.x) >= lv.first[li + 1]) ++li;
    const int base = (static_cast<int>(blockIdx.x) - lv.first[li]) * kTile + static_cast<int>(threadIdx.x) * kItems;
    int par[kItems];
    uint64_t c0 = 0, c1 = 0;
    for (int i = 0; i < kItems; ++i) {
        par[i] = base + i < lv.ncell[li] ? static_cast<int>(cellkey[lv.cell_off[li] + base + i] & 7u) : -1;
        if (par[i] >= 4) c1 += 1ull << (16 * (par[i] - 4));
        else if (par[i] >= 0) c0 += 1ull << (16 * par[i]);
    }
    uint64_t tot;
    uint64_t e0 = block_exclusive_scan<uint64_t>(c0, sh, tot);
    uint64_t e1 = block_exclusive_scan<uint64_t>(c1, sh, tot);
    for (int i = 0; i < kItems; ++i) {
        if (par[i] < 0) break;
        uint64_t& e = par[i] >= 4 ? e1 : e0;
        const int sft = 16 * (par[i] & 3);
        const int at = counts[blockIdx.x * 8 + par[i]] + static_cast<int>((e >> sft) & 0xffffu);
        e += 1ull << sft;
        order[lv.cell_off[li] + at] = base + i;
    }
}

inline unsigned blocks_for(int64_t n) { return static_cast<unsigned>((n + kBlock - 1) / kBlock); }

// Occupied M2L slots of one level counted per (parity, slot): counts[8][189].
__global__ __launch_bounds__(kBlock) void k_m2l_slot_counts(int ncell, const uint64_t* __restrict__ keys,
                                                           const int32_t* __restrict__ slots,
                                                           unsigned long long* __restrict__ counts) {
    __shared__ unsigned int bins[8 * kFarSlots];
    for (int j = threadIdx.x; j < 8 * kFarSlots; j += blockDim.x) bins[j] = 0u;
    __syncthreads();
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < ncell) {
        const int par = static_cast<int>(keys[i] & 7u);
        for (int j = 0; j < kFarSlots; ++j)
            if (slots[static_cast<int64_t>(i) * kFarSlots + j] >= 0) atomicAdd(&bins[par * kFarSlots + j], 1u);
    }
    __syncthreads();
    for (int j = threadIdx.x; j < 8 * kFarSlots; j += blockDim.x)
        if (bins[j]) atomicAdd(&counts[j], static_cast<unsigned long long>(bins[j]));
}

// P2P work items of the big leaves: ceil(count / kP2PItem) items of
// consecutive targets per leaf with more than kP2PBig particles.
template <int ITEM>
__global__ __launch_bounds__(kBlock) void k_p2p_item_counts(int nleaf, const int32_t* __restrict__ lstart,
                                                           int32_t* __restrict__ cnt) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nleaf) return;
    const int m = lstart[i + 1] - lstart[i];
    cnt[i] = m > kP2PBig ? (m + ITEM - 1) / ITEM : 0;
}

template <int ITEM>
__global__ __launch_bounds__(kBlock) void k_p2p_items(int nleaf, const int32_t* __restrict__ lstart,
                                                     const int32_t* __restrict__ off, int2* __restrict__ items) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nleaf) return;
    const int m = lstart[i + 1] - lstart[i];
    if (m <= kP2PBig) return;
    const int k = (m + ITEM - 1) / ITEM;
    for (int q = 0; q < k; ++q) items[off[i] + q] = make_int2(i, lstart[i] + q * ITEM);
}

// Sort key of a big-leaf P2P work item: the items are taken costliest first,
// so the grid ends on small items instead of waiting for a large one taken
// late.  Cost = targets x sources the item visits: its own leaf and every
// neighbour (ordered pairs), or for the mutual kernel its own leaf, its small
// neighbours and its big forward neighbours (the backward ones are skipped).
// Keys ascend with falling cost; the padding past the item count sorts last.
template <int ITEM, bool MUTUAL>
__global__ __launch_bounds__(kBlock) void k_p2p_item_cost(int64_t cap, const int32_t* __restrict__ nitems,
                                                         const int2* __restrict__ items,
                                                         const int32_t* __restrict__ lstart,
                                                         const int32_t* __restrict__ slots, uint64_t* __restrict__ keys,
                                                         int32_t* __restrict__ vals) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= cap) return;
    uint64_t key = 0xFFFFFFFFull;
    if (i < *nitems) {
        const int2 it = items[i];
        const int leaf = it.x;
        int64_t src = lstart[leaf + 1] - lstart[leaf];
        for (int s = 0; s < kNbrSlots; ++s) {
            const int nb = slots[static_cast<int64_t>(leaf) * kNbrSlots + s];
            if (nb < 0) continue;
            const int sz = lstart[nb + 1] - lstart[nb];
            if (!MUTUAL || sz <= kP2PBig || s < kNbrForward) src += sz;
        }
        const int64_t tc = min(static_cast<int64_t>(ITEM), static_cast<int64_t>(lstart[leaf + 1] - it.y));
        const uint64_t cost = min(static_cast<uint64_t>(tc * src), 0xFFFFFFFEull);
        key = 0xFFFFFFFEull - cost;
    }
    keys[i] = key;
    vals[i] = static_cast<int32_t>(i);
}

__global__ __launch_bounds__(kBlock) void k_gather_items(int64_t cap, const int32_t* __restrict__ nitems,
                                                        const int32_t* __restrict__ idx, const int2* __restrict__ in,
                                                        int2* __restrict__ out) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= cap || i >= *nitems) return;
    out[i] = in[idx[i]];
}

// Sorts the work items (count on the device, at most cap) costliest first, a
// stable sort: equal costs keep the leaf order.  A work item's results (and
// the mutual kernel's slots) follow from its leaf and first target, not from
// its place in the list, so the order changes no sum.
template <int ITEM, bool MUTUAL>
int sort_p2p_items(Context* c, int2* items, const int32_t* nitems, int64_t cap) {
    if (cap <= 1) return HFMM_OK;
    HFMM_TRY(ensure(c, c->d_itemkeys, sizeof(uint64_t) * 2 * static_cast<size_t>(cap)));
    HFMM_TRY(ensure(c, c->d_itemidx, sizeof(int32_t) * 2 * static_cast<size_t>(cap)));
    HFMM_TRY(ensure(c, c->d_items_tmp, sizeof(int2) * static_cast<size_t>(cap)));
    uint64_t* ik = c->d_itemkeys.as<uint64_t>();
    int32_t* iv = c->d_itemidx.as<int32_t>();
    prof_begin(c, "p2p_items");
    hipLaunchKernelGGL((k_p2p_item_cost<ITEM, MUTUAL>), dim3(blocks_for(cap)), dim3(kBlock), 0, c->stream, cap, nitems,
                       items, c->d_leafstart.as<int32_t>(), c->d_p2p.as<int32_t>(), ik, iv);
    prof_end(c);
    HFMM_TRY(check_launch(c, "p2p_items"));
    bool swapped = false;
    HFMM_TRY(radix_sort(c, ik, iv, ik + cap, iv + cap, cap, 32, swapped));
    if (swapped) iv += cap;
    HFMM_HIP(c, hipMemcpyAsync(c->d_items_tmp.ptr, items, sizeof(int2) * static_cast<size_t>(cap),
                               hipMemcpyDeviceToDevice, c->stream));
    prof_begin(c, "p2p_items");
    hipLaunchKernelGGL(k_gather_items, dim3(blocks_for(cap)), dim3(kBlock), 0, c->stream, cap, nitems, iv,
                       c->d_items_tmp.as<int2>(), items);
    prof_end(c);
    return check_launch(c, "p2p_items");
}

// Slot tables of the mutual mixed P2P.  A work item of big leaf A (tile t of
// kP2PMutualItem targets) evaluates A against its big forward neighbours
// (slots s < 13) once for both sides; the source-side sums for the particles
// of neighbour B go to B's slot csoff[B][12 - s] + t, A being B's backward
// neighbour in slot 25 - s.  Per big leaf B: the 13 offsets (one per backward
// slot 13..25, -1 when that neighbour is absent or small) and units[B] =
// (number of slots) x (particles of B) entries.
// An item of the FP64 kernel is taken in parts[A] parts of about part_pairs
// pairs, each a range of the sources of A itself and of its big forward
// neighbours: one wave would need 14 ms for a central item of a Plummer set of
// 120,000 particles at height 6 (256 targets, 70,000 sources).  Part 0 writes
// the targets' results, each further part a slot of A's own, after those of the
// backward neighbours.  Few items leave most of the 4,096 waves idle behind the
// longest ones, so that they go in parts of 2^14 pairs, a chunk or two of 64
// sources: near field with its combination in us, 2^14 / 2^18 / ordered pairs: 8
// items (3,000 Plummer, h6) 101 / 220 / 133; 256 (30,000 on a line, h9) 51 / 78 / 50;
// about 700 (120k Plummer, h6) 1,450 / 1,652 / 4,914; 2,500 (400k Plummer, h7)
// 2,842 / 3,066 / 8,739; 8,000 (1M uniform, h5) 3,781 / 3,470 / 5,428.
inline int64_t part_pairs(int64_t items) { return int64_t(1) << (items <= 4096 ? 14 : 18); }

__global__ __launch_bounds__(kBlock) void k_colslot_counts(int nleaf, const int32_t* __restrict__ lstart,
                                                           const int32_t* __restrict__ slots, int64_t part_pairs,
                                                           int32_t* __restrict__ csoff, int64_t* __restrict__ units,
                                                           int32_t* __restrict__ parts) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nleaf) return;
    const int m = lstart[i + 1] - lstart[i];
    int run = 0;
    for (int b = 0; b < kNbrForward; ++b) {
        int o = -1;
        const int a = slots[static_cast<int64_t>(i) * kNbrSlots + kNbrForward + b];
        if (m > kP2PBig && a >= 0) {
            const int na = lstart[a + 1] - lstart[a];
            if (na > kP2PBig) {
                o = run;
                run += (na + kP2PMutualItem - 1) / kP2PMutualItem;
            }
        }
        csoff[static_cast<int64_t>(i) * kNbrForward + b] = o;
    }
    int k = 1;
    if (part_pairs && m > kP2PBig) {
        int64_t src = m;
        for (int b = 0; b < kNbrForward; ++b) {
            const int a = slots[static_cast<int64_t>(i) * kNbrSlots + b];
            const int na = a < 0 ? 0 : lstart[a + 1] - lstart[a];
            if (na > kP2PBig) src += na;
        }
        k = static_cast<int>(min(static_cast<int64_t>(kP2PMaxParts), 1 + src * min(m, kP2PMutualItem) / part_pairs));
    }
    parts[i] = k;
    units[i] = static_cast<int64_t>(run + k - 1) * m;
}

// The claims of the FP64 kernel, item kP2PMaxParts + part, in the items' order
// (costliest first): parts per item, then their places after a scan.  Claims of
// kP2PMaxParts parts for every item, most of them empty, came to 3.3 ns per item
// and part on the one counter: 4.1 of the 8.2 ms of 2M uniform particles at height
// 6 (10,562 items).
__global__ __launch_bounds__(kBlock) void k_item_parts(int64_t cap, const int32_t* __restrict__ nitems,
                                                      const int2* __restrict__ items, const int32_t* __restrict__ parts,
                                                      int32_t* __restrict__ cnt) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < cap) cnt[i] = i < *nitems ? parts[items[i].x] : 0;
}

__global__ __launch_bounds__(kBlock) void k_item_claims(int64_t cap, const int32_t* __restrict__ nitems,
                                                       const int2* __restrict__ items, const int32_t* __restrict__ parts,
                                                       const int32_t* __restrict__ off, int32_t* __restrict__ claims) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= cap || i >= *nitems) return;
    const int k = parts[items[i].x];
    for (int p = 0; p < k; ++p) claims[off[i] + p] = static_cast<int32_t>(i) * kP2PMaxParts + p;
}

// Both and the scan between them by one workgroup, for few items (claims has room
// for every part): three launches were 50 of the 280 us of a build of 32 leaves.
constexpr int64_t kClaimsOne = 2 * kTile;

__global__ __launch_bounds__(kBlock) void k_claims_one(const int32_t* __restrict__ nitems, const int2* __restrict__ items,
                                                      const int32_t* __restrict__ parts, int32_t* __restrict__ claims,
                                                      int32_t* __restrict__ total) {
    __shared__ int32_t sh[kBlock];
    const int n = *nitems;
    int32_t at = 0;
    for (int i0 = 0; i0 < n; i0 += kTile) {
        int32_t k[kItems], sum = 0;
        const int i = i0 + static_cast<int>(threadIdx.x) * kItems;
        for (int r = 0; r < kItems; ++r) {
            k[r] = i + r < n ? parts[items[i + r].x] : 0;
            sum += k[r];
        }
        int32_t tot;
        int32_t to = at + block_exclusive_scan<int32_t>(sum, sh, tot);
        for (int r = 0; r < kItems; ++r)
            for (int p = 0; p < k[r]; ++p) claims[to++] = (i + r) * kP2PMaxParts + p;
        at += tot;
    }
    if (threadIdx.x == 0) *total = at;
}

}  // namespace

int m2l_slot_counts(Context* c, int level, unsigned long long* counts) {
    const int64_t nc = c->ncell[level];
    HFMM_TRY(zero_device(c, counts, sizeof(unsigned long long) * 8 * kFarSlots));
    if (nc == 0) return HFMM_OK;
    hipLaunchKernelGGL(k_m2l_slot_counts, dim3(blocks_for(nc)), dim3(kBlock), 0, c->stream, static_cast<int>(nc),
                       c->d_cellkey.as<uint64_t>() + c->lvl_off[level],
                       c->d_m2l.as<int32_t>() + static_cast<size_t>(c->m2l_off[level]) * kFarSlots, counts);
    return check_launch(c, "m2l_slot_counts");
}

int update_charges_device(Context* c, int rhs) {
    prof_begin(c, "gather_charges");
    hipLaunchKernelGGL(k_gather_charges, dim3(blocks_for(c->n)), dim3(kBlock), 0, c->stream, c->n,
                       c->d_perm.as<int32_t>(), c->q + static_cast<size_t>(rhs) * c->n,
                       c->d_sorted.as<double>() + 3 * c->n);
    prof_end(c);
    return check_launch(c, "gather_charges");
}

int gather_all_charges(Context* c, bool f32) {
    const int64_t npad = (c->n + 7) & ~int64_t(7);  // chunk starts 64-byte aligned
    HFMM_TRY(ensure(c, c->d_qall, (f32 ? sizeof(float) : sizeof(double)) * static_cast<size_t>(npad) * c->nrhs));
    RhsChunk ch[HFMM_MAX_RHS];
    const int nch = rhs_chunks(c->nrhs, ch);
    prof_begin(c, "gather_charges");
    for (int k = 0; k < nch; ++k) {
        if (f32)
            hipLaunchKernelGGL(k_gather_charge_chunk<float>, dim3(blocks_for(c->n)), dim3(kBlock), 0, c->stream, c->n,
                               c->d_perm.as<int32_t>(), c->q, ch[k].r0, ch[k].R,
                               c->d_qall.as<float>() + npad * ch[k].r0);
        else
            hipLaunchKernelGGL(k_gather_charge_chunk<double>, dim3(blocks_for(c->n)), dim3(kBlock), 0, c->stream,
                               c->n, c->d_perm.as<int32_t>(), c->q, ch[k].r0, ch[k].R,
                               c->d_qall.as<double>() + npad * ch[k].r0);
    }
    prof_end(c);
    return check_launch(c, "gather_charges");
}

int build_tree_device(Context* c) {
    const int64_t n = c->n;
    const int h = c->height();  // of the virtual tree
    const int L = h - 1;
    const int Lloc = c->P.tree_height - 1;  // leaf level inside one set
    const int top = c->top();
    if (n <= 0) return fail(c, HFMM_ERR_ARG, "no particles");
    if (n > (int64_t(1) << 30)) return fail(c, HFMM_ERR_ARG, "more than 2^30 particles");
    HFMM_TRY(ensure(c, c->d_keys, sizeof(uint64_t) * n));
    HFMM_TRY(ensure(c, c->d_keys2, sizeof(uint64_t) * n));
    HFMM_TRY(ensure(c, c->d_perm, sizeof(int32_t) * n));
    HFMM_TRY(ensure(c, c->d_vals2, sizeof(int32_t) * n));
    HFMM_TRY(ensure(c, c->d_count, sizeof(int64_t) * 24));
    // what the host reads once: the error flag, the big leaves, the cells of each level
    HFMM_TRY(ensure(c, c->d_flags, sizeof(int32_t) * (2 + kMaxLevels)));
    int32_t* info = c->d_flags.as<int32_t>();
    HFMM_HIP(c, hipMemsetAsync(info, 0, sizeof(int32_t) * 2, c->stream));

    // 1. keys (boxCorner = center + (-(width/2)), FGroupTree.hpp:183)
    const double half = c->P.box_width / 2;
    const double leafw = c->P.box_width / static_cast<double>(1 << Lloc);
    prof_begin(c, "morton");
    hipLaunchKernelGGL(k_morton, dim3(blocks_for(n)), dim3(kBlock), 0, c->stream, n, c->x, c->y, c->z,
                       c->P.box_center[0] + (-half), c->P.box_center[1] + (-half), c->P.box_center[2] + (-half),
                       c->P.box_width, leafw, Lloc, c->nsets > 1 ? c->d_setoff.as<int64_t>() : nullptr, c->nsets,
                       c->d_keys.as<uint64_t>(), c->d_perm.as<int32_t>(), info);
    prof_end(c);
    HFMM_TRY(check_launch(c, "morton"));

    // 2. stable sort by key (ties keep the input order)
    bool swapped = false;
    HFMM_TRY(radix_sort(c, c->d_keys.as<uint64_t>(), c->d_perm.as<int32_t>(), c->d_keys2.as<uint64_t>(),
                        c->d_vals2.as<int32_t>(), n, 3 * L, swapped));
    if (swapped) {
        std::swap(c->d_keys, c->d_keys2);
        std::swap(c->d_perm, c->d_vals2);
    }
    const uint64_t* keys = c->d_keys.as<uint64_t>();

    // 3. cells per level, and on the host
    const int64_t ntiles = (n + kTile - 1) / kTile;
    HFMM_TRY(ensure(c, c->d_scan_part, sizeof(int32_t) * static_cast<size_t>(ntiles) * (L - top + 1)));
    int32_t* counts = c->d_scan_part.as<int32_t>();
    prof_begin(c, "levels");
    hipLaunchKernelGGL(k_level_counts, dim3(static_cast<unsigned>(ntiles)), dim3(kBlock), 0, c->stream, n, keys, top, L,
                       ntiles, counts, info + 1);
    hipLaunchKernelGGL(k_level_scan, dim3(L - top + 1), dim3(kBlock), 0, c->stream, ntiles, counts, info + 2);
    prof_end(c);
    HFMM_TRY(check_launch(c, "levels"));
    int32_t h_info[2 + kMaxLevels] = {0};
    HFMM_HIP(c, hipMemcpyAsync(h_info, info, sizeof(int32_t) * (2 + L - top + 1), hipMemcpyDeviceToHost, c->stream));
    HFMM_HIP(c, hipStreamSynchronize(c->stream));
    if (h_info[0]) return fail(c, HFMM_ERR_OUTSIDE_BOX, "a particle lies outside the simulation box");
    TreeLevels lv{};
    lv.top = top;
    lv.leaf = L;
    int64_t off = 0, cs = 0;
    for (int l = 0; l < kMaxLevels; ++l) c->ncell[l] = 0;
    for (int l = 0; l <= L; ++l) {
        c->lvl_off[l] = c->m2l_off[l] = lv.lvl_off[l] = off;
        if (l < top) continue;
        c->ncell[l] = lv.ncell[l] = h_info[2 + l - top];
        off += c->ncell[l];
        c->cs_off[l] = lv.cs_off[l] = cs;
        cs += c->ncell[l] + 1;
    }
    c->lvl_off[L + 1] = off;
    c->total_cells = off;
    const int64_t nl = c->ncell[L];

    // 4. sorted particle SoA
    // kSortedPad doubles after the four SoA arrays: the big-leaf P2P reads whole
    // blocks of sources past a leaf's end (and masks them)
    HFMM_TRY(ensure(c, c->d_sorted, sizeof(double) * (4 * n + kSortedPad)));
    HFMM_TRY(ensure(c, c->d_iperm, sizeof(int32_t) * n));
    prof_begin(c, "gather");
    hipLaunchKernelGGL(k_gather_particles, dim3(blocks_for(n)), dim3(kBlock), 0, c->stream, n, c->d_perm.as<int32_t>(),
                       c->x, c->y, c->z, c->q, c->d_sorted.as<double>(), c->d_iperm.as<int32_t>());
    prof_end(c);
    HFMM_TRY(check_launch(c, "gather"));

    // 5. cell keys, leaf and child ranges
    HFMM_TRY(ensure(c, c->d_cellkey, sizeof(uint64_t) * static_cast<size_t>(off)));
    HFMM_TRY(ensure(c, c->d_leafstart, sizeof(int32_t) * (nl + 1)));
    HFMM_TRY(ensure(c, c->d_pleaf, sizeof(int32_t) * n));
    HFMM_TRY(ensure(c, c->d_childstart, sizeof(int32_t) * static_cast<size_t>(cs)));
    prof_begin(c, "levels");
    hipLaunchKernelGGL(k_level_cells, dim3(static_cast<unsigned>(ntiles)), dim3(kBlock), 0, c->stream, n, keys, lv,
                       ntiles, counts, c->d_cellkey.as<uint64_t>(), c->d_childstart.as<int32_t>(),
                       c->d_leafstart.as<int32_t>(), c->d_pleaf.as<int32_t>());
    prof_end(c);
    HFMM_TRY(check_launch(c, "levels"));

    // 6. dense Morton -> cell tables for the levels with at most 2^24 cells, then
    // the P2P slots of the leaves and the M2L slots of levels top..h-1
    int64_t dense_total = 0;
    int64_t dense_off[kMaxLevels];
    for (int l = top; l <= L; ++l) {
        dense_off[l] = -1;
        if (3 * l <= 24) {
            dense_off[l] = dense_total;
            dense_total += int64_t(1) << (3 * l);
        }
    }
    HFMM_TRY(ensure(c, c->d_dense, sizeof(int32_t) * static_cast<size_t>(dense_total + 1)));
    HFMM_HIP(c, hipMemsetAsync(c->d_dense.ptr, 0xFF, sizeof(int32_t) * static_cast<size_t>(dense_total), c->stream));
    SlotLevels sl{}, leaf{};
    for (int l = top; l <= L; ++l) {
        const int i = sl.nlev++;
        sl.ix[i].keys = c->d_cellkey.as<uint64_t>() + c->lvl_off[l];
        sl.ix[i].n = static_cast<int>(c->ncell[l]);
        sl.ix[i].dense = dense_off[l] >= 0 ? c->d_dense.as<int32_t>() + dense_off[l] : nullptr;
        sl.lim[i] = 1 << (l - c->set_levels);
        sl.cell_off[i] = c->lvl_off[l];
        sl.first[i + 1] = sl.first[i] + static_cast<int>((c->ncell[l] + kSlotCells - 1) / kSlotCells);
    }
    leaf.nlev = 1;
    leaf.ix[0] = sl.ix[sl.nlev - 1];
    leaf.lim[0] = sl.lim[sl.nlev - 1];
    leaf.first[1] = sl.first[sl.nlev] - sl.first[sl.nlev - 1];
    HFMM_TRY(ensure(c, c->d_p2p, sizeof(int32_t) * static_cast<size_t>(nl) * kNbrSlots));
    HFMM_TRY(ensure(c, c->d_m2l, sizeof(int32_t) * static_cast<size_t>(off) * kFarSlots));
    prof_begin(c, "dense_index");
    hipLaunchKernelGGL(k_dense_index, dim3(sl.first[sl.nlev]), dim3(64), 0, c->stream, sl);
    prof_end(c);
    HFMM_TRY(check_launch(c, "dense_index"));
    prof_begin(c, "p2p_lists");
    hipLaunchKernelGGL((k_cell_slots<kNbrSlots, false>), dim3(leaf.first[1]), dim3(kBlock), 0, c->stream, leaf,
                       c->d_slotpos.as<int16_t>(), c->d_p2p.as<int32_t>());
    prof_end(c);
    HFMM_TRY(check_launch(c, "p2p_lists"));
    prof_begin(c, "m2l_lists");
    hipLaunchKernelGGL((k_cell_slots<kFarSlots, true>), dim3(sl.first[sl.nlev]), dim3(kBlock), 0, c->stream, sl,
                       c->d_slotpos.as<int16_t>(), c->d_m2l.as<int32_t>());
    prof_end(c);
    HFMM_TRY(check_launch(c, "m2l_lists"));

    // 7. work items of the big leaves (slot 12 of d_count: their number)
    const int64_t nbig = h_info[1];
    c->p2p_items_cap = nbig > 0 ? n / kP2PItem + nbig : 0;
    if (c->p2p_items_cap > 0) {
        HFMM_TRY(ensure(c, c->d_p2pitems, sizeof(int2) * static_cast<size_t>(c->p2p_items_cap)));
        HFMM_TRY(ensure(c, c->d_flags, sizeof(int32_t) * static_cast<size_t>(nl + 1)));
        HFMM_TRY(ensure(c, c->d_scan, sizeof(int32_t) * static_cast<size_t>(nl + 1)));
        prof_begin(c, "p2p_items");
        hipLaunchKernelGGL(k_p2p_item_counts<kP2PItem>, dim3(blocks_for(nl)), dim3(kBlock), 0, c->stream, static_cast<int>(nl),
                           c->d_leafstart.as<int32_t>(), c->d_flags.as<int32_t>());
        prof_end(c);
        HFMM_TRY(check_launch(c, "p2p_items"));
        HFMM_TRY(exclusive_scan<int32_t>(c, c->d_flags.as<int32_t>(), c->d_scan.as<int32_t>(), nl, p2p_item_count(c),
                                         "p2p_items"));
        prof_begin(c, "p2p_items");
        hipLaunchKernelGGL(k_p2p_items<kP2PItem>, dim3(blocks_for(nl)), dim3(kBlock), 0, c->stream, static_cast<int>(nl),
                           c->d_leafstart.as<int32_t>(), c->d_scan.as<int32_t>(), c->d_p2pitems.as<int2>());
        prof_end(c);
        HFMM_TRY(check_launch(c, "p2p_items"));
        // the ordered big-leaf kernels take the items at a fixed stride: costliest
        // first spreads the large ones over the waves
        HFMM_TRY((sort_p2p_items<kP2PItem, false>(c, c->d_p2pitems.as<int2>(), p2p_item_count(c), c->p2p_items_cap)));
    }
    c->tree_built = true;
    c->evaluated = false;
    c->p2p_mutual = false;
    c->order_built = false;
    c->m2l_asked = 0;
    if (c->p2p_items_cap > 0) HFMM_TRY(build_p2p_mutual_tables(c, nbig));
    return HFMM_OK;
}

// The cells of every level by child index, for the M2L kernels that read them so
// (bfloat16 tiles, global SVD), once per tree.
int ensure_parity_order(Context* c) {
    if (c->order_built) return HFMM_OK;
    ParityLevels lv{};
    for (int l = c->top(); l < c->height(); ++l) {
        const int i = lv.nlev++;
        lv.cell_off[i] = c->lvl_off[l];
        lv.ncell[i] = static_cast<int>(c->ncell[l]);
        lv.level[i] = l;
        lv.first[i + 1] = lv.first[i] + static_cast<int>((c->ncell[l] + kTile - 1) / kTile);
    }
    HFMM_TRY(ensure(c, c->d_order, sizeof(int32_t) * static_cast<size_t>(c->total_cells)));
    HFMM_TRY(ensure(c, c->d_pcount, sizeof(int32_t) * 8 * kMaxLevels));
    HFMM_TRY(ensure(c, c->d_hist, sizeof(int32_t) * 8 * static_cast<size_t>(lv.first[lv.nlev])));
    int32_t* counts = c->d_hist.as<int32_t>();
    prof_begin(c, "parity");
    hipLaunchKernelGGL(k_parity_counts, dim3(lv.first[lv.nlev]), dim3(kBlock), 0, c->stream, lv,
                       c->d_cellkey.as<uint64_t>(), counts);
    hipLaunchKernelGGL(k_parity_scan, dim3(lv.nlev), dim3(64), 0, c->stream, lv, counts, c->d_pcount.as<int32_t>());
    hipLaunchKernelGGL(k_parity_order, dim3(lv.first[lv.nlev]), dim3(kBlock), 0, c->stream, lv,
                       c->d_cellkey.as<uint64_t>(), counts, c->d_order.as<int32_t>());
    prof_end(c);
    HFMM_TRY(check_launch(c, "parity"));
    c->order_built = true;
    return HFMM_OK;
}

// Bytes that the first evaluation of the built tree takes beside what the context
// has: expansions, results, and the M2L's least workspace (FP64 products: a step
// of rows, 1 KB per cell, partial locals, up to 4, and what the pages round up; tiles:
// multipoles in FP32).
static size_t evaluation_needs(const Context* c) {
    const auto lacks = [](const DevBuf& b, size_t bytes) { return bytes > b.bytes ? bytes - b.bytes : 0; };
    const size_t exp = sizeof(double) * static_cast<size_t>(c->total_cells + 1) * c->LD;
    const size_t values = sizeof(double) * static_cast<size_t>(c->n) * c->nrhs;
    const size_t work = static_cast<size_t>(c->total_cells) * 6144;
    const size_t own = c->d_m2lC.bytes + c->d_m2lacc.bytes;
    return lacks(c->d_M, exp) + lacks(c->d_L, exp) + lacks(c->d_res_sorted, 4 * values) + lacks(c->d_res, 4 * values) +
           lacks(c->d_field, 3 * values) + (work > own ? work - own : 0);
}

int build_p2p_mutual_tables(Context* c, int64_t nbig) {
    c->p2p_mutual = false;
    const int64_t nl = c->ncell[c->height() - 1];
    const int32_t* lstart = c->d_leafstart.as<int32_t>();
    c->p2p_items_m_cap = c->n / kP2PMutualItem + nbig;
    HFMM_TRY(ensure(c, c->d_p2pitems_m, sizeof(int2) * static_cast<size_t>(c->p2p_items_m_cap)));
    HFMM_TRY(ensure(c, c->d_flags, sizeof(int32_t) * static_cast<size_t>(nl + 1)));
    HFMM_TRY(ensure(c, c->d_scan, sizeof(int32_t) * static_cast<size_t>(nl + 1)));
    prof_begin(c, "p2p_items");
    hipLaunchKernelGGL(k_p2p_item_counts<kP2PMutualItem>, dim3(blocks_for(nl)), dim3(kBlock), 0, c->stream,
                       static_cast<int>(nl), lstart, c->d_flags.as<int32_t>());
    prof_end(c);
    HFMM_TRY(check_launch(c, "p2p_items"));
    HFMM_TRY(exclusive_scan<int32_t>(c, c->d_flags.as<int32_t>(), c->d_scan.as<int32_t>(), nl,
                                     p2p_mutual_item_count(c), "p2p_items"));
    prof_begin(c, "p2p_items");
    hipLaunchKernelGGL(k_p2p_items<kP2PMutualItem>, dim3(blocks_for(nl)), dim3(kBlock), 0, c->stream,
                       static_cast<int>(nl), lstart, c->d_scan.as<int32_t>(), c->d_p2pitems_m.as<int2>());
    prof_end(c);
    HFMM_TRY(check_launch(c, "p2p_items"));
    HFMM_TRY((sort_p2p_items<kP2PMutualItem, true>(c, c->d_p2pitems_m.as<int2>(), p2p_mutual_item_count(c),
                                                    c->p2p_items_m_cap)));
    HFMM_TRY(ensure(c, c->d_csoff, sizeof(int32_t) * static_cast<size_t>(nl) * kNbrForward));
    HFMM_TRY(ensure(c, c->d_csbase, sizeof(int64_t) * static_cast<size_t>(nl + 1)));
    HFMM_TRY(ensure(c, c->d_csparts, sizeof(int32_t) * static_cast<size_t>(nl)));
    int64_t* base = c->d_csbase.as<int64_t>();
    prof_begin(c, "p2p_items");
    hipLaunchKernelGGL(k_colslot_counts, dim3(blocks_for(nl)), dim3(kBlock), 0, c->stream, static_cast<int>(nl), lstart,
                       c->d_p2p.as<int32_t>(), is_mixed(c) ? 0 : part_pairs(c->p2p_items_m_cap), c->d_csoff.as<int32_t>(), base, c->d_csparts.as<int32_t>());
    prof_end(c);
    HFMM_TRY(check_launch(c, "p2p_items"));
    HFMM_TRY(exclusive_scan<int64_t>(c, base, base, nl, p2p_mutual_units(c), "p2p_items"));
    const int64_t cap = c->p2p_items_m_cap;
    const bool one = cap <= kClaimsOne;
    if (!is_mixed(c)) {
        if (one) HFMM_TRY(ensure(c, c->d_claims, sizeof(int32_t) * kP2PMaxParts * static_cast<size_t>(cap)));
        else HFMM_TRY(ensure(c, c->d_scan, sizeof(int32_t) * static_cast<size_t>(cap)));
        prof_begin(c, "p2p_items");
        if (one) {
            hipLaunchKernelGGL(k_claims_one, dim3(1), dim3(kBlock), 0, c->stream, p2p_mutual_item_count(c),
                               c->d_p2pitems_m.as<int2>(), c->d_csparts.as<int32_t>(), c->d_claims.as<int32_t>(), p2p_claim_count(c));
        } else {
            hipLaunchKernelGGL(k_item_parts, dim3(blocks_for(cap)), dim3(kBlock), 0, c->stream, cap, p2p_mutual_item_count(c),
                               c->d_p2pitems_m.as<int2>(), c->d_csparts.as<int32_t>(), c->d_scan.as<int32_t>());
        }
        prof_end(c);
        HFMM_TRY(check_launch(c, "p2p_items"));
        if (!one)
            HFMM_TRY(exclusive_scan<int32_t>(c, c->d_scan.as<int32_t>(), c->d_scan.as<int32_t>(), cap, p2p_claim_count(c), "p2p_items"));
    }
    int64_t counts[2] = {0, 0};  // units, claims
    HFMM_HIP(c, hipMemcpyAsync(counts, p2p_mutual_units(c), sizeof(counts), hipMemcpyDeviceToHost, c->stream));
    HFMM_HIP(c, hipStreamSynchronize(c->stream));
    const int64_t units = counts[0];
    // base[nl] = the total, so a leaf's slot count is (base[i+1] - base[i]) / n_i
    HFMM_HIP(c, hipMemcpyAsync(base + nl, p2p_mutual_units(c), sizeof(int64_t), hipMemcpyDeviceToDevice, c->stream));
    const size_t bytes = (is_mixed(c) ? sizeof(float) : sizeof(double)) * 4 * static_cast<size_t>(units > 0 ? units : 1);
    if (bytes > c->d_cpart.bytes) {
        size_t free_b = 0, total_b = 0;
        HFMM_HIP(c, hipMemGetInfo(&free_b, &total_b));
        free_b += c->d_cpart.bytes;
        const size_t later = evaluation_needs(c);
        // ordered-pair kernel instead
        if (later > free_b || bytes > free_b / 4 || bytes > free_b - later) return HFMM_OK;
    }
    HFMM_TRY(ensure(c, c->d_cpart, bytes));
    if (!is_mixed(c)) c->p2p_claims = static_cast<int32_t>(counts[1]);
    if (!is_mixed(c) && !one) {
        HFMM_TRY(ensure(c, c->d_claims, sizeof(int32_t) * static_cast<size_t>(c->p2p_claims)));
        prof_begin(c, "p2p_items");
        hipLaunchKernelGGL(k_item_claims, dim3(blocks_for(cap)), dim3(kBlock), 0, c->stream, cap, p2p_mutual_item_count(c),
                           c->d_p2pitems_m.as<int2>(), c->d_csparts.as<int32_t>(), c->d_scan.as<int32_t>(),
                           c->d_claims.as<int32_t>());
        prof_end(c);
        HFMM_TRY(check_launch(c, "p2p_items"));
    }
    c->cpart_units = units;
    c->p2p_mutual = true;
    return HFMM_OK;
}

}  // namespace hfmm

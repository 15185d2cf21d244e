// m2l_plan.hpp -- host side of the FP64 M2L (m2l_f64.hip): the rows of the
// products and their places in a target's compressed expansions C.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace hfmm {

constexpr int kTau = 56;       // offsets (|x|, |y|, |z|), far field
constexpr int kTauDummy = 56;  // of the rows that fill the last row block

// Byte offset of a lane without a partner, past the end of every buffer, plus
// the place of its row in a target's C (below 1 MiB, not negative).
constexpr uint32_t kNowhere = 0xFFF00000u;
constexpr size_t kBufferMax = kNowhere;  // bytes

// One of the 56 offsets: its position in the 7^3 cube, first row and rank.
struct TauInfo {
    int32_t pos, row0, rank, pad;
};

// One row of the products: its offset |pos|, its place in a target's C (bytes,
// variant 0), and the bytes that a negative sign of each coordinate adds (0:
// only one sign, or none, belongs to the offset).
struct __attribute__((aligned(16))) RowInfo {
    uint32_t tau, off;
    uint16_t sign[3], pad;
};

// A target's C: row block by row block, in it per offset [variant][rows of the
// offset in the block]; a variant per pair of signs that a target of one parity
// has on an axis (|x| = 1, 2: both; 3: one, by its parity; 0: none).  rboff:
// bytes before each row block.  The rows that fill the last block lie at the end
// of C, so that their place in a part of the rows (off minus the bytes before the
// part) is not negative: added to kNowhere, off = 0 gave an address before
// kNowhere, inside a buffer that reaches nearly that far.
inline void row_layout(const TauInfo (&tau)[kTau], int nrb, std::vector<RowInfo>& rows, std::vector<int>& rboff) {
    rows.assign(static_cast<size_t>(nrb) * 16, RowInfo{kTauDummy, 0, {0, 0, 0}, 0});
    for (int t = 0; t < kTau; ++t)
        for (int r = 0; r < ((tau[t].rank + 3) & ~3); ++r) rows[tau[t].row0 + r].tau = static_cast<uint32_t>(t);
    rboff.assign(nrb + 1, 0);
    int off = 0;
    for (int b = 0; b < nrb; ++b) {
        rboff[b] = off;
        for (int r = 0; r < 16;) {
            const int t = static_cast<int>(rows[16 * b + r].tau);
            int e = r;
            while (e < 16 && static_cast<int>(rows[16 * b + e].tau) == t) ++e;
            if (t != kTauDummy) {
                const int v[3] = {tau[t].pos / 49 - 3, (tau[t].pos / 7) % 7 - 3, tau[t].pos % 7 - 3};
                int bytes = 8 * (e - r);
                uint16_t sign[3] = {0, 0, 0};
                for (int a = 0; a < 3; ++a)
                    if (v[a] == 1 || v[a] == 2) sign[a] = static_cast<uint16_t>(bytes), bytes *= 2;
                for (int q = r; q < e; ++q) {
                    RowInfo& ri = rows[16 * b + q];
                    ri.off = static_cast<uint32_t>(off + 8 * (q - r));
                    for (int a = 0; a < 3; ++a) ri.sign[a] = sign[a];
                }
                off += bytes;
            }
            r = e;
        }
    }
    rboff[nrb] = off;
    for (RowInfo& ri : rows)
        if (ri.tau == kTauDummy) ri.off = static_cast<uint32_t>(off);
}

// Two column tiles per workgroup (32 cells) reuse the operators but take 1.7
// times as long as one (1,000 uniform particles, order 7: 354 against 205 us), so
// they pay where they need fewer rounds of the 256 CUs: 585 cells, order 8, 575
// against 338 us; 4,681 cells, order 5 139 / 154, order 8 595 / 711; 37,449 cells,
// order 6 1,239 / 1,400.
inline bool two_tiles(int64_t ncell) {
    const int64_t one = (ncell + 16 * 256 - 1) / (16 * 256), two = (ncell + 32 * 256 - 1) / (32 * 256);
    return 17 * two < 10 * one;
}

// Bytes that a context's workspace may take of `want`, with free_bytes left on the
// device, `own` bytes in the context's workspace and `held` in all workspaces of the
// process there: what it has, and its share of a quarter of the memory that is
// free or in workspaces, so that several contexts together leave three
// quarters to everything else.  Where that quarter is used up, a quarter of what
// is free up to kRoomMin or a sixteenth of `want`: 16 parts at most.
constexpr size_t kRoomMin = size_t(256) << 20;

inline size_t workspace_room(size_t want, size_t own, size_t held, size_t free_bytes) {
    const size_t quarter = (free_bytes + held) / 4, others = held - own;
    size_t room = std::max(own, quarter > others ? quarter - others : 0);
    room = std::max(room, std::min(std::max(want / 16, kRoomMin), (free_bytes + own) / 4));
    return std::min(want, room);
}

// The rows in parts of whole steps (`step` row blocks): part i is row blocks cut[i] ..
// cut[i + 1] - 1.  All in one part where their C fits `room` and a launch takes
// max_part row blocks, else parts whose C fits beside acc_bytes of partial locals,
// of one step at least.  Returns the bytes of C.
inline size_t cut_rows(const std::vector<int>& rboff, int step, int max_part, int64_t ncell, size_t acc_bytes, size_t room,
                       std::vector<int>& cut) {
    const int nrb = static_cast<int>(rboff.size()) - 1;
    const auto bytes = [&](int from, int to) { return static_cast<size_t>(rboff[to] - rboff[from]) * ncell; };
    if (nrb > max_part || bytes(0, nrb) > room) room = room > acc_bytes ? room - acc_bytes : 0;
    cut.assign(1, 0);
    size_t most = 0;
    while (cut.back() < nrb) {
        const int b = cut.back();
        int e = std::min(b + step, nrb);
        while (e < nrb && e + step - b <= max_part && bytes(b, std::min(e + step, nrb)) <= room) e = std::min(e + step, nrb);
        most = std::max(most, bytes(b, e));
        cut.push_back(e);
    }
    return most;
}

}  // namespace hfmm

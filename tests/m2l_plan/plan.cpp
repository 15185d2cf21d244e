// The host side of the FP64 M2L (csrc/m2l_plan.hpp) as C functions, for
// tests/m2l_plan/__init__.py.
#include "../../scalfmm_amd/csrc/m2l_plan.hpp"

using namespace hfmm;

extern "C" {

uint32_t plan_nowhere() { return kNowhere; }

// The rows for 56 ranks: row blocks, and per row its offset |pos| (56: filler),
// place in C and largest place with its signs; rboff [blocks + 1].  Returns the row
// blocks (the arrays hold 256).
int plan_rows(const int32_t* rank, uint32_t* tau_of, uint32_t* off, uint32_t* last, int32_t* rboff) {
    TauInfo tau[kTau];
    int n = 0, row = 0;
    for (int x = 0; x < 4; ++x)
        for (int y = 0; y < 4; ++y)
            for (int z = 0; z < 4; ++z) {
                if (x < 2 && y < 2 && z < 2) continue;
                tau[n] = TauInfo{((x + 3) * 7 + y + 3) * 7 + z + 3, row, rank[n], 0};
                row += (rank[n++] + 3) & ~3;
            }
    const int nrb = ((row + 15) / 16 + 1) & ~1;
    std::vector<RowInfo> rows;
    std::vector<int> ro;
    row_layout(tau, nrb, rows, ro);
    for (int i = 0; i < 16 * nrb; ++i) {
        tau_of[i] = rows[i].tau;
        off[i] = rows[i].off;
        last[i] = rows[i].off + rows[i].sign[0] + rows[i].sign[1] + rows[i].sign[2];
    }
    for (int b = 0; b <= nrb; ++b) rboff[b] = ro[b];
    return nrb;
}

int plan_two_tiles(int64_t ncell) { return two_tiles(ncell); }

uint64_t plan_room(uint64_t want, uint64_t own, uint64_t held, uint64_t free_bytes) {
    return workspace_room(want, own, held, free_bytes);
}

// Parts of the rows: their first row blocks into cut, and the end; the bytes of C.
uint64_t plan_cut(const int32_t* rboff, int nrb, int step, int max_part, int64_t ncell, uint64_t acc, uint64_t room,
                  int32_t* cut, int* parts) {
    std::vector<int> c;
    const uint64_t bytes = cut_rows(std::vector<int>(rboff, rboff + nrb + 1), step, max_part, ncell, acc, room, c);
    for (size_t i = 0; i < c.size(); ++i) cut[i] = c[i];
    *parts = static_cast<int>(c.size()) - 1;
    return bytes;
}

}  // extern "C"

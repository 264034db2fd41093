// dmc_plan.h -- host rules of the engine that need no device: what makes two
// passes the same pass, how the cells' rows are grouped, and how many blocks a
// launch takes.
#pragma once
#include <algorithm>
#include <cstdint>
#include <string>
#include <vector>

namespace tmc {

// Everything that a pass's launches depend on besides what they read from
// device memory (fields, iso-values, geometry): a captured pass is replayed for
// passes of an equal key only.
struct PassShape {
    int64_t field_type, flags;
    int64_t sweep_rows, row_form, waves, groups;   // the sweep's tiling, the cells' groups
    int64_t grid_cap, sweep_waves;
    int64_t acap, vcap, qcap, reccap;
    int64_t generic, small_colouring;
    int64_t buf_epoch;
    std::vector<int32_t> dims;                     // nx, ny, nz of each volume
};

inline std::string pass_key(const PassShape& s) {
    const int64_t head[] = {s.field_type, s.flags,  s.sweep_rows, s.row_form, s.waves,   s.groups,
                            s.grid_cap,   s.sweep_waves, s.acap,  s.vcap,     s.qcap,    s.reccap,
                            s.generic,    s.small_colouring, s.buf_epoch, (int64_t)s.dims.size()};
    std::string k(reinterpret_cast<const char*>(head), sizeof(head));
    // (each axis whole: packed into one word, axes above 2^21 points ran into
    // each other)
    k.append(reinterpret_cast<const char*>(s.dims.data()), s.dims.size() * sizeof(int32_t));
    return k;
}

// (row, segment)s per wave of k_cells and k_tmc_cells, 2^shift: from their total
// (enough waves to fill the chip come first, cells per wave second), and small
// enough that padding every volume to whole groups adds at most an eighth to
// the lists (1 KB per (row, segment)).  k_cells with 1 / 2 / 4 / 8 / 16 of them
// per wave, us: 32^3 (961 in all) 4.6 / 4.6 / 5.2 / 6.4 / 8.0; 201x174x149
// (25,752) 17 / 13 / 13 / 18 / 29; 301x257x283 (144,384) 107 / 68 / 48 / 39 /
// 36; 1024^3 (4.2 M) 1606 / 1008 / 799 / 620 / 511.  Padded to 16 whatever the
// volumes, a pass over 20,000 volumes of 2^3 points held 443 MB instead of 44.
constexpr int kMaxGroupShift = 4;
constexpr int64_t in_groups(int64_t rs, int shift) {
    return ((rs + ((int64_t)1 << shift) - 1) >> shift) << shift;
}
inline int group_shift(const std::vector<int64_t>& rs) {
    int64_t total = 0;
    for (int64_t x : rs) total += x;
    int shift = total >= (1 << 16) ? kMaxGroupShift : total >= (1 << 13) ? 2 : 0;
    for (; shift > 0; shift--) {
        int64_t padded = 0;
        for (int64_t x : rs) padded += in_groups(x, shift);
        if (padded - total <= total / 8) break;
    }
    return shift;
}

// Blocks of a launch over n items, per_block of them a block and turn: at most
// grid_cap (the caller's, dmc_launch) and, where a kernel has a limit of its own,
// at most that (0: none).
inline int64_t blocks_for(int64_t n, int64_t per_block, int64_t limit, int64_t grid_cap) {
    const int64_t cap = limit > 0 ? std::min(limit, grid_cap) : grid_cap;
    return std::max<int64_t>(1, std::min((n + per_block - 1) / per_block, cap));
}

}  // namespace tmc

// dmc_plan.h -- host rules of the engine that need no device: what makes two
// passes the same pass.
#pragma once
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

}  // namespace tmc

// When a tape with automatic checkpointing records its forward run.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace lbm_amd {

// Device memory that one allocation of `bytes` may take.
inline size_t allocated(size_t bytes) {
    constexpr size_t granule = size_t{2} << 20;
    return (bytes + granule - 1) / granule * granule;
}

// A record of nsteps steps of `step` bytes each is kept where it takes at most
// a quarter of the device's memory and half of what is free, and leaves room
// for `rest`: everything else that the tape allocates, so that a tape which
// fits with checkpoints is not refused for its record.
inline bool record_fits(uint64_t nsteps, size_t step, size_t rest, size_t free_bytes, size_t total_bytes) {
    if (step == 0 || nsteps > std::min(total_bytes / 4, free_bytes / 2) / step) return false;
    return allocated(nsteps * step) + rest <= free_bytes;
}

// `rest` of a single domain's tape: the initial field, two mu buffers and the
// gradients and target (fp64).
inline size_t tape_rest(size_t field_bytes, size_t plane_elems, int q, size_t calc_bytes, size_t near_cells,
                        size_t target_cells) {
    return allocated(field_bytes) + 2 * allocated(plane_elems * static_cast<size_t>(q) * calc_bytes) +
           allocated(8 * plane_elems) + allocated(24 * std::max<size_t>(near_cells, 1)) + allocated(24 * target_cells);
}

}  // namespace lbm_amd

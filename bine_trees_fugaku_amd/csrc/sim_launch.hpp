// sim_launch.hpp -- arguments of one simulation pass (sim.hip), shared with the host side.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace bine {

// A run of slices launched together: workgroups of one size and LDS need.
struct SimBin {
    uint32_t first, count, threads, lds;
};

struct SimLaunch {
    const void *cases, *classes;
    const void *slices;  // per workgroup of sim_class: class, first dimension | last + 1 << 8
    SimBin bins[3];
    uint32_t n_bins;
    const void *count_blocks, *scan_blocks;  // of the classes without slices
    uint32_t n_count_blocks, n_scan_blocks;
    bool zero;  // some class is counted by several workgroups: its statistics (and counters in memory) start at zero
    uint32_t* mult;
    uint64_t mult_len;
    uint32_t ncls;
    uint32_t *max_hops, *max_mult;
    uint64_t* sum_mult;
};

hipError_t launch_sim(const SimLaunch& a, hipStream_t st);
hipError_t sim_lds_limit(int device, uint32_t* bytes);

}  // namespace bine

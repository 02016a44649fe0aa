// vz_path.h -- plain launches (vzLaunch) as persistent path tracing: the
// workspace a context keeps for them and the launch itself.
#pragma once
#include "vz_engine.h"

namespace vz {

// Buffers kept by a context between launches, freed with it.  One launch
// uses them at a time (the context's mutex is held until the launch has
// finished on its stream).
struct PathWork {
    char* paths = nullptr;      // seeds and radiances of one chunk of passes
    size_t paths_bytes = 0;
    char* pixels = nullptr;     // sums and camera seeds carried from chunk to chunk
    size_t pixels_bytes = 0;
    unsigned long long* stats = nullptr;    // device: per k_path workgroup
    unsigned long long* h_stats = nullptr;  // pinned: their totals, written by k_path_resolve
    Event t0, t1;
    uint32_t grid_lds = 0, grid_mem = 0;    // resident k_path workgroups by variant
};

void path_free(PathWork* w);
// Renders one frame and waits for it.
vzStatus path_launch(vzContext ctx, const vzScene_st* scene, const vzLaunchParams& p, hipStream_t st, RunResult* res);

}  // namespace vz

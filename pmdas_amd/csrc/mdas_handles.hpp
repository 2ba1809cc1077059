// The opaque handle types of the C ABI and helpers shared by the host files.
#pragma once
#include <string>

#include "mdas.h"
#include "mdas_internal.hpp"
#include "scenes.hpp"

struct mdas_grid {
    mdas::Grid g;
};

struct mdas_scene {
    mscene::Params host;
    void* dev = nullptr;
};

namespace mdas {
// Sets the calling thread's last error message and returns `code`.
int set_error(int code, const std::string& msg);
// Copies the device counters of a grid to its host mirror (synchronising).
int sync_grid(Grid& g, hipStream_t st);
// The largest leaf extents of a fresh initial grid (after initial sampling).
void initial_extents(Grid& g);
// What a run's last kernel, a single pass or a report left of the counters,
// once it has finished.
void take_counters(Grid& g);
// Appends the rows of the passes before `done`, which have finished, to
// g.pstats_host (at most kHostRows of them since the last call).
void take_pass_rows(Grid& g, int done);
}  // namespace mdas

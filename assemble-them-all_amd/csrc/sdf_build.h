// Mesh -> signed distance grid on the GPU (the role of sdfgen::make_level_set3).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include "levelset.h"

namespace atac {

struct LsArgs {
    const float* x;           // 3 * nv vertex coordinates
    const uint32_t* tri;      // 3 * nf vertex indices
    int64_t nf;
    float o[3];               // grid origin (node (0, 0, 0))
    float dx, dy, dz;
    int32_t ni, nj, nk;
    int32_t band;             // exact band, in cells
    float phi0;               // initial (upper-bound) distance
    // per node, first (distance bits << 32) | triangle, the band's minimum; then the
    // sweeps' state: (tag << 32) | word, see ls_sweep_kernel
    unsigned long long* best;
    float* phi;               // per node: distance, then signed distance
    ls::Tri* tris;            // per triangle: its vertices and what its distances share
    int32_t* count;           // per node: x-ray crossings in (i - 1, i]
    int32_t* sync;            // kLsSync words: tiles handed out per sweep, and the give-up flag
};
constexpr int kLsSweeps = 16, kLsGaveUp = kLsSweeps, kLsSync = kLsSweeps + 1;

// Launches the whole construction on `st`: band distances and crossing counts,
// 2 x 8 fast-sweeping passes (one launch each), signs. sync[kLsGaveUp] is set when
// a sweep waited for a neighbour in vain (its values are then wrong).
hipError_t ls_build(const LsArgs& a, hipStream_t st);

}  // namespace atac

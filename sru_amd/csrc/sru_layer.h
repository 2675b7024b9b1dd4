// What the entry point of a whole layer hands to the kernels behind it.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sru_amd {

// One time step (layer_step.hip): rows (rows, inner) times weight (inner, cols).
struct StepParams {
    const void *x, *weight;
    const void *wc, *bias, *c0, *scale_x, *skip;
    const uint8_t *pad;
    void *h, *c_last;      // h: the product itself when it is the projection
    int64_t cols, Dp;
    int32_t rows, inner, act;
    uint32_t small16;
};

constexpr int kStepMaxRows = 64;   // four tiles of 16 rows share a weight operand
// 32 cells per workgroup, 32 inner indices per matrix instruction
inline bool step_sizes_ok(int64_t rows, int64_t Dp, int64_t inner, int64_t n_proj) {
    return rows <= kStepMaxRows && Dp % 32 == 0 && inner % 32 == 0 && n_proj % 32 == 0 && inner <= (1 << 24);
}
hipError_t launch_layer_step(const StepParams &p, const StepParams *proj, bool half, int k, int skip, hipStream_t st);

}  // namespace sru_amd

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

// Whole sequences with the weights in registers (layer_rows.hip): x (L * B, inner) times weight
// (inner, Dp * k).
struct RowsParams {
    const void *x, *weight;
    const void *wc, *bias, *c0, *scale_x, *skip;
    const uint8_t *pad;
    void *h, *c_last;
    int64_t B, Dp;
    int32_t L, d, dirs, inner;
    int32_t groups_per_dir;   // of 64 cells
    uint32_t small16;
};

// Walk steps per matrix tile: with two, 131072 columns are one wavefront per SIMD; up to 65536 four fill
// the chip instead (2048 steps, 65536 columns of 256 + 256 cells, f16: 627 us with two, 415 with four).
inline int rows_steps_per_tile(int64_t B, int64_t Dp) { return B * Dp <= 65536 ? 4 : 2; }
// A walk takes its 160-450 ns a step however few columns there are, two calls take time by the column:
// 2048 steps, product and scan against one kernel: 32768 columns 330-430 against 325-530 us, 49152
// columns 516-652 against 334-531 us, 131072 columns 1404 against 670 us (inner size 256) and 1432
// against 952 us (512). 256 steps at 49152 columns: 70-90 against 48-81 us; shorter walks are not
// measured.
constexpr int64_t kRowsMinColumns = 49152, kRowsMinSteps = 256;
inline bool rows_sizes_ok(int64_t L, int64_t B, int64_t d, int64_t dirs, int64_t inner, int k) {
    return d % 8 == 0 && inner % 32 == 0 && inner <= (k == 3 ? 512 : 256) && L < (1 << 30) &&
           B * d * dirs >= kRowsMinColumns && L >= kRowsMinSteps &&
           B * d * dirs < (1 << 28) && B * inner < (1 << 28);   // (a tile's addresses are 32-bit offsets from its first time)
}
hipError_t launch_layer_rows(const RowsParams &p, bool half, int k, hipStream_t st);

}  // namespace sru_amd

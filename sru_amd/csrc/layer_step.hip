// One time step of a whole layer in 16-bit weights: U = x W (or (x Wp) W) and the recurrence behind
// it, for a batch of a few rows. This is what generating text one token at a time does per layer.
//
// What bounds it: the weights have to be read once (8.4 MB per layer at 2048 features through a
// 512-wide projection, 1.6 us at the rate of a large copy); the rest of a step is launches and
// latency. A library product, a second one and a scan per layer took 9.7 + 6.4 + 3.7 us of GPU time
// (2048 features, projection 512, batch 16); here the projection is one launch and the second
// product carries the recurrence in its epilogue, so U (f32 in the accumulators) never exists in
// memory.
//
// Mapping. A workgroup of 8 wavefronts owns 16 * CW columns of the product for all rows; its
// wavefronts split the inner dimension and their partial sums meet in LDS in wavefront order. The
// weights go straight from memory to registers: a lane reads, for 8 consecutive inner indices, CW
// adjacent elements of the row-major weight (16 lanes together one contiguous row segment), and
// v_perm pairs them into MFMA operands, CW of them, of which operand i holds the columns
// m * CW + i. (CW is 6 with three streams per column and 8 with four, so that the streams of a
// column meet in one workgroup.) The rows of x are the other operand; 16 rows to a tile.
#include "sru_amd.h"

#include <hip/hip_runtime.h>

#include "sru_layer.h"
#include "sru_mfma.h"

namespace sru_amd {
namespace {

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * kBlock;
constexpr int kTileRows = 16;
constexpr int kPitch = 17;      // floats per column of a partial tile in LDS: 16 rows + 1, every bank twice per access

// STREAMS: 0 stores the product, 3 / 4 run the recurrence step on it.
// SKIP as in the scan kernels. DEPTH: MFMA steps whose loads are in flight together.
template <typename T, int CW, int NB, int STREAMS, int SKIP, int DEPTH>
__global__ void __launch_bounds__(kThreads) dense_rows(const StepParams p) {
    static_assert(CW % 2 == 0 && (STREAMS == 0 ? CW == 2 : CW == 2 * STREAMS), "16 * CW columns are 32 cells");
    constexpr int W = 16 * CW;
    __shared__ float part[kWaves][W * kPitch];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kBlock));
    const int lane = threadIdx.x % kBlock, m = lane % 16, q = lane / 16;
    const int64_t n0 = (int64_t)blockIdx.x * W;
    const int64_t N = p.cols;
    const int K = p.inner, R = p.rows;

    const int steps = K / kStepK, each = (steps + kWaves - 1) / kWaves;
    const int s0 = wave * each, s1 = min(steps, s0 + each);
    const uint16_t *wp = static_cast<const uint16_t *>(p.weight) + (int64_t)(q * 8) * N + n0 + m * CW;
    const uint16_t *xp[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)   // rows past the last repeat it and are dropped
        xp[b] = static_cast<const uint16_t *>(p.x) + (int64_t)min(b * kTileRows + m, R - 1) * K + q * 8;

    f32x4 acc[NB][CW];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < CW; ++i) acc[b][i] = f32x4{0.f, 0.f, 0.f, 0.f};

    struct Stage {
        Words<CW / 2> w[8];
        u32x4 x[NB];
    };
    for (int s = s0; s < s1; s += DEPTH) {
        Stage st[DEPTH];
#pragma unroll
        for (int t = 0; t < DEPTH; ++t) {
            const int64_t k = (int64_t)min(s + t, s1 - 1) * kStepK;   // a step past the last repeats it and is not used
#pragma unroll
            for (int r = 0; r < 8; ++r)
                st[t].w[r].v = *reinterpret_cast<const typename WordVec<CW / 2>::type *>(wp + (k + r) * N);
#pragma unroll
            for (int b = 0; b < NB; ++b) st[t].x[b] = *reinterpret_cast<const u32x4_a4 *>(xp[b] + k);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < DEPTH; ++t) {
            if (s + t < s1) {
#pragma unroll
                for (int i = 0; i < CW; ++i) {
                    const uint32_t pick = (i & 1) ? 0x07060302u : 0x05040100u;   // high or low halves of two dwords
                    u32x4 a;
#pragma unroll
                    for (int h = 0; h < 4; ++h)
                        a[h] = __builtin_amdgcn_perm(st[t].w[2 * h + 1].get(i / 2), st[t].w[2 * h].get(i / 2), pick);
#pragma unroll
                    for (int b = 0; b < NB; ++b) acc[b][i] = mfma<T>(a, st[t].x[b], acc[b][i]);
                }
            }
        }
    }

    const int cell = threadIdx.x % 32, row_in = threadIdx.x / 32;   // 32 cells x 16 rows
    const int64_t j = (int64_t)blockIdx.x * 32 + cell;
    SmallElem<T> ew1, ew2, eb1, eb2, ex;
    const bool wc16 = (p.small16 & kSmallWeightC) != 0, bias16 = (p.small16 & kSmallBias) != 0;
    const bool init16 = (p.small16 & kSmallInit) != 0, scale16 = (p.small16 & kSmallScale) != 0;
    const int Dp = (int)p.Dp;
    if constexpr (STREAMS != 0) {
        ew1.fetch(p.wc, j, wc16);
        ew2.fetch(p.wc, Dp + j, wc16);
        eb1.fetch(p.bias, j, bias16);
        eb2.fetch(p.bias, Dp + j, bias16);
        if (SKIP == 1 && p.scale_x) ex.fetch(p.scale_x, 0, scale16);
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if (b > 0) __syncthreads();
#pragma unroll
        for (int i = 0; i < CW; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[wave][((4 * q + r) * CW + i) * kPitch + m] = acc[b][i][r];
        __syncthreads();
        const int row = b * kTileRows + row_in;
        if (row >= R) continue;
        constexpr int S = STREAMS == 0 ? 1 : STREAMS;
        float u[S];
#pragma unroll
        for (int i = 0; i < S; ++i) {
            u[i] = 0.f;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) u[i] += part[w][(cell * S + i) * kPitch + row_in];
        }
        if constexpr (STREAMS == 0) {
            static_cast<uint16_t *>(p.h)[(int64_t)row * N + j] = (uint16_t)float_to_bits<T>(u[0]);
        } else {
            const int64_t at = (int64_t)row * Dp + j;
            float cur = 0.f;
            if (p.c0) {
                SmallElem<T> e0;
                e0.fetch(p.c0, at, init16);
                cur = e0.get(init16);
            }
            const float sx = (SKIP == 1 && p.scale_x) ? ex.get(scale16) : 1.0f;
            const float g1 = gate<T>(u[1], ew1.get(wc16), cur, eb1.get(bias16));
            const float g2 = gate<T>(u[2], ew2.get(wc16), cur, eb2.get(bias16));
            const float cn = (cur - u[0]) * g1 + u[0];
            const float val = p.act ? tanh_fast(cn) : cn;
            float out;
            if constexpr (SKIP != 0) {
                const float xv = SKIP == 1 ? bits_to_float<T>(static_cast<const uint16_t *>(p.skip)[at]) * sx : u[S - 1];
                out = (val - xv) * g2 + xv;
            } else {
                out = val * g2;
            }
            const bool padded = p.pad && p.pad[row] != 0;   // keeps the state and emits zero
            static_cast<uint16_t *>(p.h)[at] = (uint16_t)float_to_bits<T>(padded ? 0.f : out);
            put_last<T>(p.c_last, at, padded ? cur : cn, (p.small16 & kSmallLast) != 0);
        }
    }
}

template <typename T, int CW, int STREAMS, int SKIP, int DEPTH>
hipError_t launch_rows(const StepParams &p, hipStream_t st) {
    void *args[] = {const_cast<StepParams *>(&p)};
    // (four row tiles leave registers for half as many steps in flight)
    const void *f = p.rows <= 16   ? reinterpret_cast<const void *>(dense_rows<T, CW, 1, STREAMS, SKIP, DEPTH>)
                    : p.rows <= 32 ? reinterpret_cast<const void *>(dense_rows<T, CW, 2, STREAMS, SKIP, DEPTH>)
                                   : reinterpret_cast<const void *>(dense_rows<T, CW, 4, STREAMS, SKIP, DEPTH / 2>);
    return hipLaunchKernel(f, dim3((unsigned)(p.cols / (16 * CW))), dim3(kThreads), args, 0, st);
}

template <typename T>
hipError_t step_of(const StepParams &p, const StepParams *proj, int k, int skip, hipStream_t st) {
    // As many steps in flight as a wavefront has, where that is half as many or fewer: a stage loads all of
    // its steps, used or not. (2048 features, projection 512, batch 16, 2 steps: 6.5 us with four in
    // flight, 5.3 with two; a layer of 1024 features, projection 256: 10.9 -> 8.7.)
    const auto has = [](const StepParams &q, int n) { return q.inner <= n * kStepK * kWaves; };
    if (proj) {
        const hipError_t e = has(*proj, 4) ? launch_rows<T, 2, 0, 0, 4>(*proj, st) : launch_rows<T, 2, 0, 0, 8>(*proj, st);
        if (e != hipSuccess) return e;
    }
    if (k == 4) return launch_rows<T, 8, 4, 2, 2>(p, st);
    if (has(p, 2)) return skip == 1 ? launch_rows<T, 6, 3, 1, 2>(p, st) : launch_rows<T, 6, 3, 0, 2>(p, st);
    return skip == 1 ? launch_rows<T, 6, 3, 1, 4>(p, st) : launch_rows<T, 6, 3, 0, 4>(p, st);
}

}  // namespace

hipError_t launch_layer_step(const StepParams &p, const StepParams *proj, bool half, int k, int skip, hipStream_t st) {
    return half ? step_of<half_bits>(p, proj, k, skip, st) : step_of<bf16_bits>(p, proj, k, skip, st);
}

}  // namespace sru_amd

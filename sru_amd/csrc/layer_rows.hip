// A whole layer in 16-bit weights over long sequences: U = x W and the recurrence in one kernel, U only
// ever in registers.
//
// What bounded it: U. At 4096 steps, batch 256, 256 cells in two directions the product wrote 4.3 GB
// that the scan read again: library product + scan 1877 + 850 us (inner size 256, four streams) and
// 1877 + 816 us (512, three). Here a wavefront keeps the weights of 16 cells in registers for the
// whole walk and streams x past them: 1346 and 1858 us. What bounds it now is one wavefront's
// instruction issue: of 1484 cycles for two steps of the first, matrix cores work for 512, 855 issue
// an instruction, 467 wait for the one before it; nothing waits for memory.
//
// Mapping. The rows of a matrix tile are TT walk steps of 16 / TT batch elements; its columns are, for
// each stream, the same 16 cells. So lane (q, m) of the result holds all streams of cells 4q .. 4q+3 for
// row m: the recurrence runs on the accumulators where they are. With TT > 1 the state passes from the
// lanes of one step to those of the next through the lane-row shift of DPP, and only the two
// multiply-adds and the gate of the state are repeated for it; the output gate runs once for all rows.
// (TT trades repeated arithmetic for wavefronts: 16 columns x 16 / TT batch elements each.)
// Four wavefronts (64 cells) share the rows of x through LDS, staged in registers kAhead tiles ahead.
// A SIMD holds one wavefront (the weights take 96-256 registers), so nothing but the order of its
// instructions overlaps the matrix products of one tile with the recurrence of the tile before it:
// the recurrence is written as stages of four independent instructions with a few matrix
// instructions pinned between them. (Left to the compiler, products first and then the four cells one
// after the other, and with branches in the loop: 1461 and 2197 us.)
// The last tile ends at the last step; rows that the tile before it already had pass the state through.
#include "sru_amd.h"

#include <hip/hip_runtime.h>

#include <type_traits>

#include "sru_layer.h"
#include "sru_mfma.h"

namespace sru_amd {
namespace {

#define SRU_AMD_INLINE __attribute__((always_inline))   // for lambdas: called several times from unrolled code

constexpr int kRowWaves = 4;
constexpr int kRowThreads = kRowWaves * kBlock;
constexpr int kTileCells = 16;
constexpr int kAhead = 4;   // tiles of x in flight per thread (even: the LDS buffer index stays static)

// lanes of step t + 1 take the value of step t's lanes, all others keep `old`
template <int NB, int BANKS>
__device__ __forceinline__ float from_step_before(float old, float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, old), __builtin_bit_cast(int, v),
                                                                 0x110 + NB, 0xf, BANKS, false));   // row_shr:NB
}
// step 0's lanes take the value of the last step's
template <int NB>
__device__ __forceinline__ float from_last_step(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + NB, 0xf, 0xf, true));   // row_ror:NB
}

template <int N, int I = 0, typename F> __device__ __forceinline__ void static_for(F &&f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}

template <typename T, int K, int SKIP, int KS, int TT, bool PAD>
__global__ void __launch_bounds__(kRowThreads, 1) layer_rows(const RowsParams p) {
    constexpr int NB = 16 / TT;            // batch elements per tile
    constexpr int kUnits = KS * 4;         // 16-byte units of a staged row
    constexpr int kLoads = 16 * kUnits / kRowThreads;
    __shared__ u32x4 tile[2][16][kUnits + 1];   // (one unit of padding: 16 rows hit 64 different banks)

    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kBlock));
    const int lane = threadIdx.x % kBlock, m = lane % 16, q = lane / 16;
    // workgroups that read the same rows of x follow each other on the same XCD (8 of them in turn)
    const int groups = p.dirs * p.groups_per_dir;
    const int in_chunk = (int)(blockIdx.x / 8) % groups;
    const int64_t bg = (int64_t)(blockIdx.x / 8 / groups) * 8 + blockIdx.x % 8;
    if (bg * NB >= p.B) return;
    const int dir = in_chunk / p.groups_per_dir;
    const int cell0 = ((in_chunk % p.groups_per_dir) * kRowWaves + wave) * kTileCells;
    const int L = p.L;
    const int inner = p.inner, n = inner / kStepK;
    const int64_t B = p.B, Dp = p.Dp, b0 = bg * NB;

    for (int i = threadIdx.x; i < 2 * 16 * (kUnits + 1); i += kRowThreads) (&tile[0][0][0])[i] = u32x4{0, 0, 0, 0};

    // Rows of a (cells) come in fours, those past the last repeat the last four, as rows past the last
    // batch element repeat that: such lanes compute and store what the lane they repeat does, and the
    // body of the walk has no branch. (d is a multiple of 4.)
    const int my_cell = min(cell0 + m / 4 * 4, p.d - 4) + m % 4;
    u32x4 w[KS][K];
#pragma unroll
    for (int s = 0; s < KS; ++s) {   // (no branch: the loads of all of them are in flight together)
        const bool on = s < n;
        load_cell_weights<K>(static_cast<const uint16_t *>(p.weight), Dp * K, ((int64_t)dir * p.d + my_cell) * K, (on ? s : 0) * kStepK + q * 8, w[s]);
#pragma unroll
        for (int i = 0; i < K; ++i) w[s][i] = on ? w[s][i] : u32x4{0, 0, 0, 0};
    }
    // (in accumulation registers, where matrix operands may come from; left alone, the compiler spills
    // some there and moves them back for every product)
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int i = 0; i < K; ++i) asm volatile("" : "+a"(w[s][i]));

    // Rows of a tile: step base + t in walk order, base = i * TT but for the last tile. Addresses are a
    // uniform base (the tile's lowest time) and a 32-bit offset that a lane keeps for the whole walk.
    auto tile_base = [&](int i) SRU_AMD_INLINE { return min(i * TT, L - TT); };
    auto low_time = [&](int i) SRU_AMD_INLINE { return (int64_t)(dir ? L - TT - tile_base(i) : tile_base(i)); };
    auto row_in_tile = [&](int row) SRU_AMD_INLINE {   // rows past the last batch element repeat it
        const int t = row / NB;
        return (uint32_t)(dir ? TT - 1 - t : t) * (uint32_t)B + (uint32_t)min(b0 + row % NB, B - 1);
    };

    // staging of x
    uint32_t x_off[kLoads];
    int x_unit[kLoads];   // where it goes in LDS; units past the inner size go to the padding
#pragma unroll
    for (int l = 0; l < kLoads; ++l) {
        const int unit = threadIdx.x + l * kRowThreads, col = unit % kUnits;
        const bool on = col < n * 4;
        x_unit[l] = unit / kUnits * (kUnits + 1) + (on ? col : kUnits);
        x_off[l] = (row_in_tile(unit / kUnits) * (uint32_t)inner + (on ? col * 8 : 0)) * 2;
    }
    u32x4 stage[kAhead][kLoads];
    auto load_x = [&](int64_t offset, u32x4 (&to)[kLoads]) SRU_AMD_INLINE {
        const char *at = static_cast<const char *>(p.x) + offset;
#pragma unroll
        for (int l = 0; l < kLoads; ++l) to[l] = *reinterpret_cast<const u32x4 *>(at + x_off[l]);
    };
    auto put_x = [&](int buf, const u32x4 (&from)[kLoads]) SRU_AMD_INLINE {
#pragma unroll
        for (int l = 0; l < kLoads; ++l) (&tile[buf][0][0])[x_unit[l]] = from[l];
    };

    // this lane's row of a tile and its four cells
    const int my_step = m / NB;
    const int64_t my_b = min(b0 + m % NB, B - 1);
    const int64_t j = (int64_t)dir * p.d + min(cell0 + 4 * q, p.d - 4);
    const uint32_t pad_off = row_in_tile(m), cell_off = (pad_off * (uint32_t)Dp + (uint32_t)j) * 2;
    u32x2 skip[kAhead];
    uint32_t flag[kAhead];
    auto load_row = [&](int64_t skip_at, int64_t pad_at, u32x2 &s, uint32_t &f) SRU_AMD_INLINE {
        if constexpr (SKIP == 1) s = *reinterpret_cast<const u32x2 *>(static_cast<const char *>(p.skip) + skip_at + cell_off);
        if constexpr (PAD) f = *(p.pad + pad_at + pad_off);
    };
    // The uniform offsets of a tile. In the body of the walk they move by a constant (two scalar
    // additions); a wavefront that has its SIMD to itself pays for scalar instructions like for any other.
    const int64_t x_row = B * inner * 2, h_row = B * Dp * 2, sign = dir ? -TT : TT;

    float w1[4], w2[4], b1[4], b2[4], cin[4], sx = 1.0f;
    {
        SmallElem<T> ew1[4], ew2[4], eb1[4], eb2[4], e0[4], ex;
        const bool wc16 = (p.small16 & kSmallWeightC) != 0, bias16 = (p.small16 & kSmallBias) != 0;
        const bool init16 = (p.small16 & kSmallInit) != 0, scale16 = (p.small16 & kSmallScale) != 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            ew1[r].fetch(p.wc, j + r, wc16);
            ew2[r].fetch(p.wc, Dp + j + r, wc16);
            eb1[r].fetch(p.bias, j + r, bias16);
            eb2[r].fetch(p.bias, Dp + j + r, bias16);
            if (p.c0) e0[r].fetch(p.c0, my_b * Dp + j + r, init16);
        }
        if (SKIP == 1 && p.scale_x) ex.fetch(p.scale_x, 0, scale16);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            w1[r] = ew1[r].get(wc16);
            w2[r] = ew2[r].get(wc16);
            b1[r] = eb1[r].get(bias16);
            b2[r] = eb2[r].get(bias16);
            cin[r] = p.c0 ? e0[r].get(init16) : 0.f;
        }
        if (SKIP == 1 && p.scale_x) sx = ex.get(scale16);
    }

#pragma unroll
    for (int r = 0; r < 4; ++r) {   // the factor that turns exp into the hardware's exp2, as in gate()
        w1[r] *= kNegLog2e;
        w2[r] *= kNegLog2e;
        b1[r] *= kNegLog2e;
        b2[r] *= kNegLog2e;
    }

    constexpr int kProducts = KS * K;
    auto read_x = [&](int buf, u32x4 (&xf)[KS]) SRU_AMD_INLINE {
#pragma unroll
        for (int s = 0; s < KS; ++s) xf[s] = tile[buf][m][s * 4 + q];
    };
    // matrix instructions first .. last - 1 of a tile
    auto products = [&](const u32x4 (&xf)[KS], f32x4 (&acc)[K], auto first, auto last) SRU_AMD_INLINE {
#pragma unroll
        for (int i = first; i < last; ++i)
            acc[i % K] = mfma<T>(w[i / K][i % K], xf[i / K], i < K ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[i % K]);
    };

    constexpr int kStages = 1 + 7 * TT + 8, kFirst = 3;
    // The recurrence over tile i (its products in u) with the products of the next one between its stages.
    // (passed: leading rows that the tile before it had)
    auto recur = [&](int passed, int64_t h_at, const f32x4 (&u)[K], u32x2 s, uint32_t f, const u32x4 (&xf)[KS], f32x4 (&next)[K], auto &&middle) SRU_AMD_INLINE {
        auto stage_done = [&](auto n) SRU_AMD_INLINE {
            constexpr int S = decltype(n)::value;
            constexpr int span = kStages - kFirst;   // (the first stages cover the latency of reading x from LDS)
            if constexpr (S >= kFirst)
                products(xf, next, std::integral_constant<int, kProducts * (S - kFirst) / span>{},
                         std::integral_constant<int, kProducts * (S + 1 - kFirst) / span>{});
            __builtin_amdgcn_sched_barrier(0);
        };
        auto four = [&](auto n, auto &&op) SRU_AMD_INLINE {
#pragma unroll
            for (int r = 0; r < 4; ++r) op(r);
            stage_done(n);
        };
#define STAGE(n) std::integral_constant<int, (n)>{}
        const bool past = my_step < passed;
        const bool padded = PAD && f != 0, keep = past || padded;
        float prev[4], cn[4], a[4], e[4], dif[4], xv[4];
        four(STAGE(0), [&](int r) SRU_AMD_INLINE { a[r] = __builtin_fmaf(kNegLog2e, u[1][r], b1[r]); prev[r] = cin[r]; });
        static_for<TT>([&](auto tc) SRU_AMD_INLINE {
            constexpr int t = decltype(tc)::value, at = 1 + 7 * t;
            four(STAGE(at), [&](int r) SRU_AMD_INLINE { e[r] = __builtin_fmaf(w1[r], prev[r], a[r]); });
            four(STAGE(at + 1), [&](int r) SRU_AMD_INLINE { e[r] = __builtin_amdgcn_exp2f(e[r]); });
            four(STAGE(at + 2), [&](int r) SRU_AMD_INLINE { e[r] = 1.0f + e[r]; dif[r] = prev[r] - u[0][r]; });
            four(STAGE(at + 3), [&](int r) SRU_AMD_INLINE { e[r] = __builtin_amdgcn_rcpf(e[r]); });
            four(STAGE(at + 4), [&](int r) SRU_AMD_INLINE { cn[r] = __builtin_fmaf(dif[r], e[r], u[0][r]); });
            four(STAGE(at + 5), [&](int r) SRU_AMD_INLINE { if (PAD || passed) cn[r] = keep ? prev[r] : cn[r]; });
            if constexpr (t + 1 < TT) {
                constexpr int banks = TT == 2 ? 0xc : 2 << t;
                four(STAGE(at + 6), [&](int r) SRU_AMD_INLINE { prev[r] = from_step_before<NB, banks>(prev[r], cn[r]); });
            } else {
                four(STAGE(at + 6), [&](int r) SRU_AMD_INLINE { a[r] = __builtin_fmaf(kNegLog2e, u[2][r], b2[r]); });
            }
        });
        middle();
        constexpr int at = 1 + 7 * TT;
        four(STAGE(at), [&](int r) SRU_AMD_INLINE { e[r] = __builtin_fmaf(w2[r], prev[r], a[r]); cin[r] = from_last_step<NB>(cn[r]); });
        four(STAGE(at + 1), [&](int r) SRU_AMD_INLINE { e[r] = __builtin_amdgcn_exp2f(e[r]); });
        four(STAGE(at + 2), [&](int r) SRU_AMD_INLINE {
            e[r] = 1.0f + e[r];
            xv[r] = SKIP == 1 ? bits_to_float<T>((r & 1) ? s[r / 2] >> 16 : s[r / 2] & 0xffffu) : u[K - 1][r];
        });
        four(STAGE(at + 3), [&](int r) SRU_AMD_INLINE { e[r] = __builtin_amdgcn_rcpf(e[r]); });
        four(STAGE(at + 4), [&](int r) SRU_AMD_INLINE { if (SKIP == 1) xv[r] *= sx; });
        four(STAGE(at + 5), [&](int r) SRU_AMD_INLINE { dif[r] = cn[r] - xv[r]; });
        four(STAGE(at + 6), [&](int r) SRU_AMD_INLINE { e[r] = __builtin_fmaf(dif[r], e[r], xv[r]); if (PAD) e[r] = padded ? 0.f : e[r]; });
        uint32_t lo = pack_pair<T>(e[0], e[1]), hi = pack_pair<T>(e[2], e[3]);
        asm volatile("" : "+v"(lo), "+v"(hi));   // (else the stages above move into the branch, past the products)
        if (!passed || !past)
            *reinterpret_cast<u32x2 *>(static_cast<char *>(p.h) + h_at + cell_off) = u32x2{lo, hi};
        stage_done(STAGE(at + 7));
#undef STAGE
    };

    const int tiles = (L + TT - 1) / TT;
    // (the first loads are issued in the order of the loop: with any other, the compiler's wait for the
    // oldest of them at the head of the loop drains all)
    u32x4 first_x[2][kLoads];
    load_x(low_time(0) * x_row, first_x[0]);
    load_x(low_time(1) * x_row, first_x[1]);
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
        load_x(low_time(i + 2) * x_row, stage[(i + 2) % kAhead]);
        load_row(low_time(i) * h_row, low_time(i) * B, skip[i], flag[i]);
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();   // the zeros are in place
    put_x(0, first_x[0]);
    put_x(1, first_x[1]);
    __syncthreads();
    f32x4 acc[2][K];
    u32x4 xf[KS];
    read_x(0, xf);
    products(xf, acc[0], std::integral_constant<int, 0>{}, std::integral_constant<int, kProducts>{});
    // one tile, and the loads for later ones
    auto walk = [&](auto slot, int passed, int64_t x_at, int64_t skip_at, int64_t pad_at, int64_t h_at) SRU_AMD_INLINE {
        constexpr int a = decltype(slot)::value;
        __syncthreads();
        read_x((a + 1) & 1, xf);
        __builtin_amdgcn_sched_barrier(0);
        recur(passed, h_at, acc[a & 1], skip[a], flag[a], xf, acc[(a + 1) & 1], [&]() SRU_AMD_INLINE {
            // tile i + 2 goes where tile i was, which all have read before this tile's barrier
            put_x(a & 1, stage[(a + 2) % kAhead]);
            load_x(x_at, stage[(a + 2) % kAhead]);
        });
        load_row(skip_at, pad_at, skip[a], flag[a]);
    };
    int base = 0;
    int64_t xa = low_time(2 + kAhead) * x_row, sa = low_time(kAhead) * h_row, pa = low_time(kAhead) * B, ha = low_time(0) * h_row;
    for (; (base + 2 * kAhead + 2) * TT <= L; base += kAhead)
        static_for<kAhead>([&](auto slot) SRU_AMD_INLINE {
            asm volatile("" : "+s"(xa), "+s"(sa), "+s"(pa), "+s"(ha));   // (kept scalar: a lane adds its own 32 bits in the access)
            walk(slot, 0, xa, sa, pa, ha);
            xa += sign * x_row;
            sa += sign * h_row;
            pa += sign * B;
            ha += sign * h_row;
        });
    for (; base < tiles; base += kAhead)   // (tiles past the last pass the state through and store nothing)
        static_for<kAhead>([&](auto slot) SRU_AMD_INLINE {
            const int i = base + decltype(slot)::value;
            const int64_t later = low_time(i + kAhead);
            walk(slot, i * TT - tile_base(i), low_time(i + 2 + kAhead) * x_row, later * h_row, later * B, low_time(i) * h_row);
        });
    if (my_step == 0) {
        const bool last16 = (p.small16 & kSmallLast) != 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) put_last<T>(p.c_last, my_b * Dp + j + r, cin[r], last16);
    }
}

template <typename T, int K, int SKIP, int KS, int TT>
hipError_t launch(const RowsParams &p, hipStream_t st) {
    const int64_t batch_groups = (p.B + 16 / TT - 1) / (16 / TT);
    const int64_t blocks = (batch_groups + 7) / 8 * 8 * p.dirs * p.groups_per_dir;
    if (blocks > INT32_MAX) return hipErrorInvalidValue;
    void *args[] = {const_cast<RowsParams *>(&p)};
    const void *f = p.pad ? reinterpret_cast<const void *>(layer_rows<T, K, SKIP, KS, TT, true>)
                          : reinterpret_cast<const void *>(layer_rows<T, K, SKIP, KS, TT, false>);
    return hipLaunchKernel(f, dim3((unsigned)blocks), dim3(kRowThreads), args, 0, st);
}

template <typename T, int K, int SKIP, int KS>
hipError_t launch_steps(const RowsParams &p, int steps_per_tile, hipStream_t st) {
    return steps_per_tile == 4 ? launch<T, K, SKIP, KS, 4>(p, st) : launch<T, K, SKIP, KS, 2>(p, st);
}

template <typename T, int K, int SKIP>
hipError_t launch_inner(const RowsParams &p, int steps_per_tile, hipStream_t st) {
    if (p.inner <= 128) return launch_steps<T, K, SKIP, 4>(p, steps_per_tile, st);
    if (p.inner <= 256) return launch_steps<T, K, SKIP, 8>(p, steps_per_tile, st);
    if constexpr (K == 3) return launch_steps<T, K, SKIP, 16>(p, steps_per_tile, st);
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_layer_rows(const RowsParams &p, bool half, int k, hipStream_t st) {
    const int tt = rows_steps_per_tile(p.B, p.Dp);
    if (k == 4) return half ? launch_inner<half_bits, 4, 2>(p, tt, st) : launch_inner<bf16_bits, 4, 2>(p, tt, st);
    return half ? launch_inner<half_bits, 3, 1>(p, tt, st) : launch_inner<bf16_bits, 3, 1>(p, tt, st);
}

}  // namespace sru_amd

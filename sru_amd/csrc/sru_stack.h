// What the kernels of whole stacks share: handing results over between workgroups of one launch, and the piece of work of one
// time step or of a projection.
#pragma once

#include <hip/hip_runtime.h>

#include "sru_layer.h"
#include "sru_mfma.h"

namespace sru_amd {

typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));

constexpr int kStackWaves = 8;
constexpr int kStackThreads = kStackWaves * kBlock;
constexpr int kTileRows = 16, kCells = 32;
constexpr int kPitch = 17;      // floats per column of a partial tile in LDS: 16 rows + 1, every bank twice per access
constexpr uint32_t kNotYet = 0xffffffffu;
constexpr int kCoherent = 16;   // cache policy of a buffer access (sc1): served where all XCDs see the same
constexpr int kOutside = 1 << 30;   // a byte offset behind the end of every buffer
// Every wait ends by itself (layer_stack.hip). Should one not, a workgroup stops waiting after some seconds, and what
// it then reads are NaNs, which reach every result.
constexpr int kPatience = 1 << 22;

struct StackControl {
    int next, patience;
};
constexpr int kStackParts = kStackWaves * 2 * 16 * 6 * kPitch;   // floats of partial sums in LDS: of two row tiles, or of four narrow ones

// A workgroup's next piece of work, drawn ahead of its turn by one thread.
__device__ __forceinline__ int draw_piece(const StackParams &p) {
    return (int)(__hip_atomic_fetch_add(p.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u);   // (from kNotYet on)
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t stack_buffer(const void *base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, bytes, 0x00027000);
}
__device__ __forceinline__ uint32_t load_word(const void *at) {
    return __hip_atomic_load(static_cast<const uint32_t *>(at), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void hand_over(void *at, uint32_t word, uint32_t nan) {   // nan: for a NaN that is the pattern
    __hip_atomic_store(static_cast<uint32_t *>(at), word == kNotYet ? nan : word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// two lanes' 16-bit elements as one dword, in the even lane
__device__ __forceinline__ uint32_t pair_up(uint32_t bits) {
    const uint32_t other = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)bits, 0xB1, 0xf, 0xf, true);
    return bits | other << 16;
}
__device__ __forceinline__ uint32_t awaited(const void *at, uint32_t word, StackControl &control) {   // word: loaded before, perhaps too early
    if (word == kNotYet) {
        const int patience = *const_cast<volatile int *>(&control.patience);
        for (int spin = 0; spin < patience && word == kNotYet; ++spin) word = load_word(at);
        if (word == kNotYet) control.patience = 0;
    }
    return word;
}

// A size, again for each piece: what follows from the sizes would otherwise be computed once for all of them and held in more
// scalar registers than there are.
__device__ __forceinline__ int again(int size) {
    asm volatile("" : "+s"(size));
    return size;
}

// One piece. PROJECT: its 32 columns of the projection; otherwise its 32 cells of the layer. MANY: of many that wait at a time.
template <typename T, int CW, int NB, int DEPTH, bool PROJECT, bool MANY = false>
__device__ __forceinline__ void piece(const StackParams &p, float *parts, StackControl &control, int l, int tile, int row0, int R) {
    constexpr int W = 16 * CW;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kBlock));
    const int lane = threadIdx.x % kBlock, m = lane % 16, q = lane / 16;
    const StackLayer &layer = p.layer[l];
    const int all = again(p.rows), Dp = again(p.Dp), n_proj = again(p.n_proj);
    const int small16 = again((int)p.small16), act = again(p.act), has_skip = again(p.skip);
    const int N = PROJECT ? n_proj : 3 * Dp, K = PROJECT || !n_proj ? Dp : n_proj;
    // what the layer reads and, of a projected one, what the product reads
    const uint16_t *const outputs = reinterpret_cast<const uint16_t *>(p.exchange + p.outputs_at);
    const uint16_t *const in = l == 0 ? static_cast<const uint16_t *>(p.x) : outputs + (int64_t)(l - 1) * all * Dp;
    uint16_t *const projected = reinterpret_cast<uint16_t *>(p.exchange) + (int64_t)l * all * n_proj;
    const bool own = PROJECT || !n_proj;
    const bool wait = !own || l > 0;      // (the caller's own input may hold the pattern)
    const __amdgpu_buffer_rsrc_t xs = own ? stack_buffer(in, all * Dp * 2) : stack_buffer(projected, all * n_proj * 2);

    const int steps = K / kStepK, each = (steps + kStackWaves - 1) / kStackWaves;
    const int s0 = wave * each, s1 = min(steps, s0 + each);
    const int n0 = tile * W;
    const __amdgpu_buffer_rsrc_t ws = stack_buffer(PROJECT ? layer.weight_proj : layer.weight, K * N * 2);
    const int pitch = N * 2, w0 = q * 8 * pitch + (n0 + m * CW) * 2;
    int at[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)   // rows past the last repeat it and are dropped
        at[b] = ((row0 + min(b * kTileRows + m, R - 1)) * K + q * 8) * 2;

    f32x4 acc[NB][CW];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < CW; ++i) acc[b][i] = f32x4{0.f, 0.f, 0.f, 0.f};

    Words<CW / 2> w[DEPTH][8];
    u32x4 x[DEPTH][NB];
    // (steps past the last lie behind the end of their buffer, where loads give zeros)
    auto load_weights = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < DEPTH; ++t) {
            const int from = s + t < s1 ? (s + t) * kStepK * pitch : kOutside;
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                if constexpr (CW == 2) w[t][r].v = __builtin_amdgcn_raw_buffer_load_b32(ws, w0 + from + r * pitch, 0, 0);
                else w[t][r].v = __builtin_bit_cast(u32x3, __builtin_amdgcn_raw_buffer_load_b96(ws, w0 + from + r * pitch, 0, 0));
            }
        }
    };
    load_weights(s0);

    // the recurrence's operands, which are there already
    const int cell = threadIdx.x % kCells, row_in = threadIdx.x / kCells;   // 32 cells x 16 rows
    const int j = tile * kCells + cell;
    SmallElem<T> ew1{}, ew2{}, eb1{}, eb2{}, ex{}, e0[NB]{};
    const bool wc16 = (small16 & kSmallWeightC) != 0, bias16 = (small16 & kSmallBias) != 0;
    const bool init16 = (small16 & kSmallInit) != 0, scale16 = (small16 & kSmallScale) != 0;
    uint32_t skip[NB], pads = 0;
#pragma unroll
    for (int b = 0; b < NB; ++b) skip[b] = kNotYet;
    const auto skip_at = [&](int b) __attribute__((always_inline)) {
        return in + (int64_t)(row0 + min(b * kTileRows + row_in, R - 1)) * Dp + (j & ~1);
    };
    if constexpr (!PROJECT) {
        ew1.fetch(layer.wc, j, wc16);
        ew2.fetch(layer.wc, Dp + j, wc16);
        eb1.fetch(layer.bias, j, bias16);
        eb2.fetch(layer.bias, Dp + j, bias16);
        if (has_skip && layer.scale_x) ex.fetch(layer.scale_x, 0, scale16);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int row = min(b * kTileRows + row_in, R - 1);
            if (p.c0) e0[b].fetch(p.c0, ((int64_t)l * R + row) * Dp + j, init16);
            if (p.pad) pads |= (p.pad[row0 + row] != 0 ? 1u : 0u) << b;
        }
    }

    for (int s = s0; s < s1; s += DEPTH) {
        const int patience = *const_cast<volatile int *>(&control.patience);
        for (int spin = 0;; ++spin) {
            asm volatile("" ::: "memory");   // (the loads are made again each time)
            uint32_t most = 0;
#pragma unroll
            for (int t = 0; t < DEPTH; ++t) {
                const int from = s + t < s1 ? (s + t) * (kStepK * 2) : kOutside;
#pragma unroll
                for (int b = 0; b < NB; ++b) x[t][b] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xs, at[b] + from, 0, kCoherent));
            }
            if constexpr (!PROJECT) {   // (with the last of them what the skip term reads arrives as well, or nearly)
                if (has_skip && s == s0) {
#pragma unroll
                    for (int b = 0; b < NB; ++b) skip[b] = load_word(skip_at(b));
                }
            }
            if (!wait) break;
#pragma unroll
            for (int t = 0; t < DEPTH; ++t)
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int i = 0; i < 4; ++i) most = max(most, x[t][b][i]);
            if (__all(most != kNotYet)) break;
            if (spin >= patience) {
                control.patience = 0;
                break;
            }
            if constexpr (MANY) {   // (until one of them is there: many workgroups that ask for all keep the memory busy)
                for (; spin < patience; ++spin) {
                    asm volatile("" ::: "memory");
                    const u32x4 one = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xs, at[NB - 1] + s * (kStepK * 2), 0, kCoherent));
                    if (__all(max(max(one[0], one[1]), max(one[2], one[3])) != kNotYet)) break;
                }
            }
        }
#pragma unroll
        for (int t = 0; t < DEPTH; ++t) {
#pragma unroll
            for (int i = 0; i < CW; ++i) {
                const uint32_t pick = (i & 1) ? 0x07060302u : 0x05040100u;   // high or low halves of two dwords
                u32x4 a;
#pragma unroll
                for (int h = 0; h < 4; ++h)
                    a[h] = __builtin_amdgcn_perm(w[t][2 * h + 1].get(i / 2), w[t][2 * h].get(i / 2), pick);
#pragma unroll
                for (int b = 0; b < NB; ++b) acc[b][i] = mfma<T>(a, x[t][b], acc[b][i]);
            }
        }
        if (s + DEPTH < s1) load_weights(s + DEPTH);
    }

    const auto put_h = [&](int row, float value) __attribute__((always_inline)) {   // of the layer
        const uint32_t word = pair_up(float_to_bits<T>(value));
        if (cell & 1) return;
        const int64_t to = (int64_t)(row0 + row) * Dp + j;
        if (l + 1 == again(p.layers)) *reinterpret_cast<uint32_t *>(static_cast<uint16_t *>(p.h) + to) = word;
        else hand_over(const_cast<uint16_t *>(outputs) + (int64_t)l * all * Dp + to, word, 0x7fff7fffu);
    };
    const float sx = !PROJECT && has_skip && layer.scale_x ? ex.get(scale16) : 1.0f;
    const auto skip_of = [&](int b) __attribute__((always_inline)) {
        if (l > 0) skip[b] = awaited(skip_at(b), skip[b], control);
        else if (s0 >= s1) skip[b] = load_word(skip_at(b));
        return bits_to_float<T>(cell & 1 ? skip[b] >> 16 : skip[b] & 0xffffu) * sx;
    };
    constexpr int kAtOnce = PROJECT || NB < 2 ? NB : 2;   // row tiles between barriers
    const auto part = [&](int v, int b) __attribute__((always_inline)) { return parts + (v * kAtOnce + b % kAtOnce) * (W * kPitch); };
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if (b % kAtOnce == 0) {
            if (b > 0) __syncthreads();
#pragma unroll
            for (int g = b; g < b + kAtOnce; ++g)
#pragma unroll
                for (int i = 0; i < CW; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) part(wave, g)[((4 * q + r) * CW + i) * kPitch + m] = acc[g][i][r];
            __syncthreads();
        }
        const int row = b * kTileRows + row_in;
        if (row >= R) continue;
        constexpr int S = PROJECT ? 1 : 3;
        float u[S];
#pragma unroll
        for (int i = 0; i < S; ++i) {
            u[i] = 0.f;
#pragma unroll
            for (int v = 0; v < kStackWaves; ++v) u[i] += part(v, b)[(cell * S + i) * kPitch + row_in];
        }
        if constexpr (PROJECT) {
            const uint32_t word = pair_up(float_to_bits<T>(u[0]));
            if (!(cell & 1)) hand_over(projected + (int64_t)(row0 + row) * n_proj + j, word, 0x7fff7fffu);
        } else {
            const float cur = e0[b].get(init16);   // (zeros where there is none)
            const float g1 = gate<T>(u[1], ew1.get(wc16), cur, eb1.get(bias16));
            const float g2 = gate<T>(u[2], ew2.get(wc16), cur, eb2.get(bias16));
            const float cn = (cur - u[0]) * g1 + u[0];
            const float val = act ? tanh_fast(cn) : cn;
            float out = val * g2;
            if (has_skip) {
                const float xv = skip_of(b);
                out = (val - xv) * g2 + xv;
            }
            const bool padded = pads >> b & 1;   // keeps the state and emits zero
            put_h(row, padded ? 0.f : out);
            put_last<T>(p.c_last, ((int64_t)l * R + row) * Dp + j, padded ? cur : cn, (small16 & kSmallLast) != 0);
        }
    }
}

}  // namespace sru_amd

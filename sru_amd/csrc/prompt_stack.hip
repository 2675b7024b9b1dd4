// A short sequence of few batch rows through a stack of equal layers in 16-bit weights without gradients, in one launch: a
// prompt, each layer working on another part of it.
//
// What bounds it: layer after layer, a prompt of 512 steps through ten layers of 2048 features (projection 512) was ten serial
// walks of 21 us on 32 of 256 compute units, each behind two short products, 23 us: 427 us. Here a layer starts on the first steps
// when the layer before has done these: 286 us. 128 steps 229 -> 144, 1024 640 -> 496; 370 steps, ten layers of 256, 207 -> 93.
// What bounds it now: of the way from a layer to the next, 16 us for 64 steps, 3.7 are the projection, 7.4 the walking piece (3.0 of
// them the walk itself, 2.8 the product), the rest handing over; and once there are many chunks on their way, 25 us for each
// of them, workgroups that wait in a compute unit's only place.
//
// Pieces. A chunk is a number of time steps of all batch rows, 64 rows at the most. Per layer and chunk there are n_proj / 32
// pieces that project 32 columns each (sru_stack.h), and Dp / 64 that make U for 64 cells, float and never in memory, and walk
// the chunk's steps. A piece only reads what pieces of smaller numbers write (prompt_piece in sru_layer.h has the numbers); how they are
// drawn and how they hand results over is layer_stack.hip's.
//
// Their order. From a layer to the next it is three times as far as from a chunk to the next, which waits for a walk alone, so a
// layer's projection of a chunk is numbered with what is `stride` chunks further on in the layer before, and its walk `delay`
// chunks behind it: drawn about when it can begin, a piece holds its place for less waiting. (Along the diagonals of layer and
// chunk, a stride of one, the same prompt took 332 us, 1024 steps 560, 2048 of six layers of 512 268 -> 177; two chunks and one
// behind 334 and 554, three and two 356 and 600, four and one 317 and 488. Chunks of 32 rows best at four and two.)
//
// A walking piece: 512 inner indices of all rows pass through LDS at a time (the next ones on their way in registers); of these two
// groups of four wavefronts take one half each, and a wavefront 16 cells with their three streams, weights from memory
// straight into matrix operands, eight matrix steps ahead. The groups swap halves of their sums through LDS; one thread per
// cell and batch row walks the state; everything else of a step is done where the sums are.
#include "sru_amd.h"

#include <hip/hip_runtime.h>

#include "sru_relay.h"
#include "sru_stack.h"

namespace sru_amd {
namespace {

constexpr int kWalkCells = 64;
constexpr int kPhase = 512;                       // inner indices in LDS at a time
constexpr int kPhaseSteps = kPhase / kStepK / 2;  // matrix steps of a group in a phase
constexpr int kPitchX = kPhase * 2 + 16;          // bytes of a row in LDS: 16 rows side by side reach every bank
constexpr int kPitchWalk = kWalkCells + 2, kPitchState = kWalkCells + 4;   // elements, for the same reason

template <int TILES> struct WalkLds {   // after the product, in the place of x
    f32x4_alias swap[kStackWaves][TILES / 2 * 3][kBlock];
    f32x2_alias walk[TILES * kTileRows][kPitchWalk];          // u0 and the state gate's sum without the state
    float states[2 * TILES * kTileRows][kPitchState];         // row r: the state before row r of the chunk
};
template <int TILES> union PromptLds {
    char x[2][TILES * kTileRows * kPitchX];
    WalkLds<TILES> w;
    float parts[kStackWaves * 2 * 2 * 16 * kPitch];           // of a projecting piece of 32 rows
};

__device__ __forceinline__ void hand_over_pair(void *at, u32x2 words) {
    uint64_t v = (uint64_t)(words[1] == kNotYet ? 0x7fff7fffu : words[1]) << 32 | (words[0] == kNotYet ? 0x7fff7fffu : words[0]);
    __hip_atomic_store(static_cast<uint64_t *>(at), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u32x2 load_pair(const void *at) {
    const uint64_t v = __hip_atomic_load(static_cast<const uint64_t *>(at), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return u32x2{(uint32_t)v, (uint32_t)(v >> 32)};
}

// 64 cells of a layer over a chunk: rows row0 .. row0 + R - 1 of all
template <typename T, int TILES, bool ONE_PHASE>
__device__ __forceinline__ void walk_piece(const StackParams &p, PromptLds<TILES> &lds, StackControl &control, int l, int chunk, int tile, int row0, int R) {
    constexpr int kRows = TILES * kTileRows;
    constexpr int kAheadW = ONE_PHASE || TILES == 2 ? kPhaseSteps : 4;   // matrix steps whose weights are on their way (as registers allow)
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kBlock));
    const int group = wave / 4;
    const int lane = threadIdx.x % kBlock, m = lane % 16, q = lane / 16;
    const StackLayer &layer = p.layer[l];
    const int B = again(p.batch), all = again(p.rows), Dp = again(p.Dp), n_proj = again(p.n_proj);
    const int small16 = again((int)p.small16), act = again(p.act), has_skip = again(p.skip);
    const int K = n_proj ? n_proj : Dp, pitch = 3 * Dp * 2;
    const uint16_t *const outputs = reinterpret_cast<const uint16_t *>(p.exchange + p.outputs_at);
    const uint16_t *const in = l == 0 ? static_cast<const uint16_t *>(p.x) : outputs + (int64_t)(l - 1) * all * Dp;
    const bool wait = n_proj || l > 0;    // (the caller's own input may hold the pattern)
    const __amdgpu_buffer_rsrc_t xs = n_proj ? stack_buffer(reinterpret_cast<const uint16_t *>(p.exchange) + (int64_t)l * all * n_proj, all * n_proj * 2)
                                             : stack_buffer(in, all * Dp * 2);
    const __amdgpu_buffer_rsrc_t ws = stack_buffer(layer.weight, K * pitch);
    const int phases = ONE_PHASE ? 1 : (K + kPhase - 1) / kPhase;

    // this lane's cell as a column of the matrix steps (cells past the last repeat it and are dropped)
    const int cell0 = tile * kWalkCells + wave % 4 * 16, column = 3 * min(cell0 + m, Dp - 1), odd = column & 1;
    const int w0 = q * 8 * pitch + (column - odd) * 2;   // (three elements from a 4-byte boundary: see load_cell_weights)
    u32x2 w[kAheadW][8];
    const auto load_weights = [&](int phase, int t) __attribute__((always_inline)) {
        const int k = phase * kPhase + (group * kPhaseSteps + t) * kStepK, from = k < K ? k * pitch : kOutside;
#pragma unroll
        for (int r = 0; r < 8; ++r) w[t % kAheadW][r] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(ws, w0 + from + r * pitch, 0, 0));
    };
#pragma unroll
    for (int t = 0; t < kAheadW; ++t) load_weights(0, t);

    // rows of x on their way to LDS: a wavefront takes every eighth, a lane 16 bytes of each
    constexpr int kMine = kRows / kStackWaves;
    u32x4 stage[kMine];
    const auto load_x = [&](int phase) __attribute__((always_inline)) {
        const int k = phase * kPhase + lane * 8, from = k < K ? k * 2 : kOutside;
#pragma unroll
        for (int i = 0; i < kMine; ++i)
            stage[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xs, (row0 + min(i * kStackWaves + wave, R - 1)) * K * 2 + from, 0, kCoherent));
    };
    const auto arrived = [&]() __attribute__((always_inline)) {
        uint32_t most = 0;
#pragma unroll
        for (int i = 0; i < kMine; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) most = max(most, stage[i][e]);
        return __all(most != kNotYet);
    };
    const auto await_x = [&](int phase) __attribute__((always_inline)) {   // loaded once before
        if (!wait) return;
        const int patience = *const_cast<volatile int *>(&control.patience);
        for (int spin = 0; !arrived(); ++spin) {
            if (spin >= patience) {
                control.patience = 0;
                break;
            }
            for (; spin < patience; ++spin) {   // (until one row is there: many workgroups that ask for all keep the memory busy)
                asm volatile("" ::: "memory");
                const int k = phase * kPhase + lane * 8, from = k < K ? k * 2 : kOutside;
                const u32x4 one = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xs, (row0 + min((kMine - 1) * kStackWaves + wave, R - 1)) * K * 2 + from, 0, kCoherent));
                if (__all(max(max(one[0], one[1]), max(one[2], one[3])) != kNotYet)) break;
            }
            load_x(phase);
        }
    };
    const auto put_x = [&](int phase) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kMine; ++i) *reinterpret_cast<u32x4_alias *>(&lds.x[phase & 1][(i * kStackWaves + wave) * kPitchX + lane * 16]) = stage[i];
    };

    // After the product a lane has four adjacent cells of row m of two of the row tiles; their operands, and what the chain's
    // threads start from, are asked for here.
    constexpr int kOwn = TILES / 2;
    const int first = cell0 + 4 * q, within = wave % 4 * 16 + 4 * q;   // (Dp is a multiple of 32: all four are there or none)
    const bool there = first < Dp;
    const int cells = min(first, Dp - 4), chunks = again(p.chunks);
    SmallElem<T> ew2[4], eb1[4], eb2[4], ex{}, ew1{}, e0{};
    const bool wc16 = (small16 & kSmallWeightC) != 0, bias16 = (small16 & kSmallBias) != 0, init16 = (small16 & kSmallInit) != 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        ew2[i].fetch(layer.wc, Dp + cells + i, wc16);
        eb1[i].fetch(layer.bias, cells + i, bias16);
        eb2[i].fetch(layer.bias, Dp + cells + i, bias16);
    }
    if (has_skip && layer.scale_x) ex.fetch(layer.scale_x, 0, (small16 & kSmallScale) != 0);
    const int j = tile * kWalkCells + (int)threadIdx.x % kWalkCells, jc = min(j, Dp - 1);   // the chain's cell
    ew1.fetch(layer.wc, jc, wc16);
    u32x2 skip[kOwn];
    uint32_t pads = 0;
    const auto row_of = [&](int b) __attribute__((always_inline)) { return (group * kOwn + b) * kTileRows + m; };
    const auto skip_at = [&](int b) __attribute__((always_inline)) { return in + (int64_t)(row0 + min(row_of(b), R - 1)) * Dp + cells; };
    if (p.pad) {
#pragma unroll
        for (int b = 0; b < kOwn; ++b) pads |= (p.pad[row0 + min(row_of(b), R - 1)] != 0 ? 1u : 0u) << b;
    }

    f32x4 acc[TILES][3];
#pragma unroll
    for (int b = 0; b < TILES; ++b)
#pragma unroll
        for (int i = 0; i < 3; ++i) acc[b][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    load_x(0);
    await_x(0);
    const auto load_skip = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < kOwn; ++b) skip[b] = has_skip ? load_pair(skip_at(b)) : u32x2{0, 0};
    };
    if constexpr (ONE_PHASE) load_skip();
    put_x(0);
    __syncthreads();
    for (int phase = 0; phase < phases; ++phase) {
        const bool more = phase + 1 < phases;
        if (more) load_x(phase + 1);
        const char *const rows = &lds.x[phase & 1][m * kPitchX + group * (kPhaseSteps * kStepK * 2) + q * 16];
#pragma unroll
        for (int t = 0; t < kPhaseSteps; ++t) {
            u32x4 a[3], x[TILES];
            u32x2 (&now)[8] = w[t % kAheadW];
#pragma unroll
            for (int b = 0; b < TILES; ++b) x[b] = *reinterpret_cast<const u32x4_alias *>(rows + b * (kTileRows * kPitchX) + t * (kStepK * 2));
#pragma unroll
            for (int r = 0; r < 8; ++r) now[r] = u32x2{__builtin_amdgcn_alignbit(now[r][1], now[r][0], odd * 16), now[r][1] >> (odd * 16)};
#pragma unroll
            for (int s = 0; s < 3; ++s)
#pragma unroll
                for (int h = 0; h < 4; ++h)   // the low or high halves of two dwords
                    a[s][h] = __builtin_amdgcn_perm(now[2 * h + 1][s / 2], now[2 * h][s / 2], (s & 1) ? 0x07060302u : 0x05040100u);
            if (t + kAheadW < kPhaseSteps) load_weights(phase, t + kAheadW);
            else if (more) load_weights(phase + 1, t + kAheadW - kPhaseSteps);
#pragma unroll
            for (int b = 0; b < TILES; ++b)
#pragma unroll
                for (int s = 0; s < 3; ++s) acc[b][s] = mfma<T>(a[s], x[b], acc[b][s]);
        }
        if (more) {
            await_x(phase + 1);
            put_x(phase + 1);
            __syncthreads();
        }
    }

    if constexpr (!ONE_PHASE) load_skip();   // (for want of registers before)
    // (the chain's first state, of the first batch rows that a thread has)
    float *const kept = reinterpret_cast<float *>(p.exchange + p.states_at);   // the state behind each chunk but the last
    const int n = R / B;
    const auto state_at = [&](int b) __attribute__((always_inline)) { return kept + ((int64_t)(l * (chunks - 1) + chunk - 1) * B + b) * Dp + jc; };
    uint32_t early = kNotYet;
    if (chunk > 0 && (int)threadIdx.x < kWalkCells * B) early = load_word(state_at(threadIdx.x / kWalkCells));

    __syncthreads();   // x has been read
#pragma unroll
    for (int b = 0; b < kOwn; ++b)
#pragma unroll
        for (int s = 0; s < 3; ++s) lds.w.swap[wave][b * 3 + s][lane] = group == 0 ? acc[kOwn + b][s] : acc[b][s];
    __syncthreads();
    f32x4 u2[kOwn];
#pragma unroll
    for (int b = 0; b < kOwn; ++b) {
        f32x4 u[3];
#pragma unroll
        for (int s = 0; s < 3; ++s) {   // (the first half of a phase first, whoever adds)
            const f32x4 mine = group == 0 ? acc[b][s] : acc[kOwn + b][s], other = lds.w.swap[wave ^ 4][b * 3 + s][lane];
            u[s] = mine + other;
        }
        u2[b] = u[2];
        f32x4 pairs[2];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float sum = __builtin_fmaf(kNegLog2e, u[1][i], kNegLog2e * eb1[i].get(bias16));
            const uint32_t bits = __builtin_bit_cast(uint32_t, sum);
            pairs[i / 2][i % 2 * 2] = u[0][i];
            pairs[i / 2][i % 2 * 2 + 1] = __builtin_bit_cast(float, (pads >> b & 1) ? kRelayPadded : bits == kRelayPadded ? bits ^ 1u : bits);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) *reinterpret_cast<f32x4_alias *>(&lds.w.walk[row_of(b)][within + 2 * i]) = pairs[i];
    }
    __syncthreads();

    // the state's chain, a thread to a cell of a batch row
    for (int c = threadIdx.x; c < kWalkCells * B && j < Dp; c += kStackThreads) {
        const int b = c / kWalkCells, cell = c % kWalkCells;   // (the same cell each time)
        __builtin_amdgcn_s_setprio(3);
        const int64_t of_layer = ((int64_t)l * B + b) * Dp + j;
        float state = 0.f;
        if (chunk > 0) {
            state = __builtin_bit_cast(float, awaited(state_at(b), early, control));
            early = kNotYet;
        } else if (p.c0) {
            e0.fetch(p.c0, of_layer, init16);
            state = e0.get(init16);
        }
        const float w1 = kNegLog2e * ew1.get(wc16);
        const f32x2_alias *from = &lds.w.walk[b][cell];
        float *to = &lds.w.states[b][cell];
        const int step_from = B * kPitchWalk, step_to = B * kPitchState;
        *to = state;
        const auto walk = [&](auto some_padded) __attribute__((always_inline)) {
            const auto step = [&](const f32x2_t op) __attribute__((always_inline)) {
                const float u0 = op[0], sum = op[1];
                const float g = sigmoid_exp2<T>(__builtin_fmaf(w1, state, sum));
                const float cn = __builtin_fmaf(state - u0, g, u0);
                state = decltype(some_padded)::value && __builtin_bit_cast(uint32_t, sum) == kRelayPadded ? state : cn;
                to += step_to;
                *to = state;
            };
            constexpr int kAhead = 8;
            int t = 0;
            if (n >= kAhead) {
                f32x2_t now[kAhead];
                const f32x2_alias *at = from;
#pragma unroll
                for (int r = 0; r < kAhead; ++r) now[r] = at[r * step_from];
                for (; t + kAhead <= n; t += kAhead) {
                    at = from + min(t + kAhead, n - kAhead) * step_from;   // (what follows the last of them is read from LDS below)
#pragma unroll
                    for (int r = 0; r < kAhead; ++r) {
                        const f32x2_t op = now[r];
                        now[r] = at[r * step_from];
                        step(op);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            for (; t < n; ++t) step(from[t * step_from]);
        };
        if (p.pad) walk(std::true_type{});
        else walk(std::false_type{});
        if (chunk + 1 < chunks)
            hand_over(state_at(b) + (int64_t)B * Dp, __builtin_bit_cast(uint32_t, state), 0x7fffffffu);
        else
            put_last<T>(p.c_last, of_layer, state, (small16 & kSmallLast) != 0);
        __builtin_amdgcn_s_setprio(0);
    }
    __syncthreads();

    const float sx = has_skip && layer.scale_x ? ex.get((small16 & kSmallScale) != 0) : 1.0f;
#pragma unroll
    for (int b = 0; b < kOwn; ++b) {
        const int row = row_of(b);
        if (row >= R || !there) continue;
        const f32x4 before = *reinterpret_cast<const f32x4_alias *>(&lds.w.states[row][within]);
        const f32x4 after = *reinterpret_cast<const f32x4_alias *>(&lds.w.states[row + B][within]);
        if (has_skip && l > 0) {
            skip[b][0] = awaited(skip_at(b), skip[b][0], control);
            skip[b][1] = awaited(skip_at(b) + 2, skip[b][1], control);
        }
        float out[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float g2 = sigmoid_exp2<T>(__builtin_fmaf(kNegLog2e * ew2[i].get(wc16), before[i], __builtin_fmaf(kNegLog2e, u2[b][i], kNegLog2e * eb2[i].get(bias16))));
            const float cn = after[i], val = act ? tanh_fast(cn) : cn;
            const float xv = bits_to_float<T>((i & 1) ? skip[b][i / 2] >> 16 : skip[b][i / 2] & 0xffffu) * sx;
            out[i] = has_skip ? (val - xv) * g2 + xv : val * g2;
            if (pads >> b & 1) out[i] = 0.f;
        }
        const u32x2 words = {pack_pair<T>(out[0], out[1]), pack_pair<T>(out[2], out[3])};
        const int64_t at = (int64_t)(row0 + row) * Dp + first;
        if (l + 1 == again(p.layers)) *reinterpret_cast<u32x2 *>(static_cast<uint16_t *>(p.h) + at) = words;
        else hand_over_pair(const_cast<uint16_t *>(outputs) + (int64_t)l * all * Dp + at, words);
    }
}

template <typename T, int TILES, bool ONE_PHASE>
__global__ void __launch_bounds__(kStackThreads) prompt_stack(const StackParams p) {
    __shared__ PromptLds<TILES> lds;
    __shared__ StackControl control;
    if (threadIdx.x == 0) control = StackControl{draw_piece(p), kPatience};
    __syncthreads();
    int number = __builtin_amdgcn_readfirstlane(control.next);
    int slot = 0, before = 0;   // pieces of earlier slots
    while (number < p.pieces) {
        int drawn = 0;
        if (threadIdx.x == 0) drawn = draw_piece(p);
        // (projecting pieces are of 32 rows: registers for all that they read)
        const PromptOrder order = {again(p.layers), again(p.chunks), again(p.stride), again(p.delay),
                                   again(p.n_proj) / kCells * (TILES / 2), again(p.projecting_last), (again(p.Dp) + kWalkCells - 1) / kWalkCells};
        const PromptPiece at = prompt_piece(order, number, slot, before);
        const int rows = again(p.steps) * again(p.batch), row0 = at.chunk * rows, R = min(rows, again(p.rows) - row0);
        if (at.project) {
            const int halves = min(TILES / 2, (R + 31) / 32), from = at.index % halves * 32;
            piece<T, 2, 2, 8, true, true>(p, lds.parts, control, at.layer, at.index / halves, row0 + from, min(R - from, 32));
        } else
            walk_piece<T, TILES, ONE_PHASE>(p, lds, control, at.layer, at.chunk, at.index, row0, R);
        // (every wavefront has read `number`: either kind of piece has a barrier, and there are no empty ones)
        if (threadIdx.x == 0) control.next = drawn;
        __syncthreads();
        number = __builtin_amdgcn_readfirstlane(control.next);
    }
}

template <typename T> const void *kernel_of(int tiles, bool one) {
    if (tiles == 2) return one ? reinterpret_cast<const void *>(prompt_stack<T, 2, true>) : reinterpret_cast<const void *>(prompt_stack<T, 2, false>);
    return one ? reinterpret_cast<const void *>(prompt_stack<T, 4, true>) : reinterpret_cast<const void *>(prompt_stack<T, 4, false>);
}

}  // namespace

hipError_t launch_prompt_stack(StackParams p, void *workspace, size_t bytes, bool half, hipStream_t st) {
    const int tiles = p.steps * p.batch <= 32 ? 2 : 4;
    const PromptOrder order = prompt_order(p);
    p.pieces = prompt_pieces(order);
    p.stride = order.stride;
    p.delay = order.delay;
    p.projecting_last = order.projecting_last;
    const hipError_t e = clear_exchange(p, workspace, bytes, st);
    if (e != hipSuccess) return e;
    void *args[] = {&p};
    const bool one = (p.n_proj ? p.n_proj : p.Dp) <= kPhase;
    const void *f = half ? kernel_of<half_bits>(tiles, one) : kernel_of<bf16_bits>(tiles, one);
    return hipLaunchKernel(f, dim3((unsigned)(p.pieces < 256 ? p.pieces : 256)), dim3(kStackThreads), args, 0, st);
}

}  // namespace sru_amd

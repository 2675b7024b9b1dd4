// Forward scan for few columns: the walk's serial chain on a wavefront of its own.
//
// What bounds it. Below about one wavefront per SIMD the time of a walk is the time of one step of
// one wavefront: 64 ns for a 16-bit lane-pair step (16 vector instructions, LDS reads, waits; 512 steps of
// 2048 columns 32.6 us on 64 of the chip's 1024 SIMDs), while the state's own dependence is a
// multiply-add, exp2, add, reciprocal and a multiply-add. Here one wavefront of a workgroup does only
// that, for 64 columns, and kRelayHelpers others do the rest: memory, conversions, the output gate.
// 512 steps of 2048 columns bf16: 33.4 -> 21 us, float 38.7 -> 26; 201 steps of 12160 columns (d = 152 or 304) 21.5 -> 13.2.
// What bounds it now: a step of the chain, 33 ns of which 27 remain when the helpers do nothing (six dependent
// instructions, two of them transcendental); a fifth of a chunk is its hand-over (chunks of 8 steps: 40 ns a
// step; of 32: no faster, for the helpers' registers).
//
// Mapping. A workgroup owns 64 adjacent columns (any directions and batch rows) and walks them in
// chunks of TC steps. Chunk j passes through the workgroup in stages, one barrier apart:
//   j      helpers write its elements, loaded A chunks earlier, to LDS as they are in memory;
//   j + 1  helpers turn them into the chain's operands (u0 and the state gate's sum without the state,
//          float) and keep the output gate's operands in registers;
//   j + 2  the chain reads its operands into registers;
//   j + 3  the chain walks the chunk and leaves the states in LDS;
//   j + 4  helpers compute the outputs of the chunk and store them.
// Memory is touched in pieces of 16 bytes; a piece never straddles a direction or a batch row where
// d is a multiple of the elements in it, so each has one time order.
//
// Padding. A padded step reaches the chain as a sentinel in place of its sum. Where a workgroup's columns
// lie in few batch rows, leading and trailing padding is not walked (as in the chunked kernels).
#pragma once

#include <type_traits>

#include "sru_scan.h"

namespace sru_amd {

typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef u32x4_t __attribute__((may_alias)) u32x4_alias;
typedef u32x2_t __attribute__((may_alias)) u32x2_alias;
typedef f32x2_t __attribute__((may_alias)) f32x2_alias;
typedef f32x4_t __attribute__((may_alias)) f32x4_alias;
typedef uint32_t __attribute__((may_alias)) u32_alias;

template <int I> using Int = std::integral_constant<int, I>;

constexpr int kRelayCols = 64, kRelayHelpers = 4, kRelaySteps = 16;
constexpr int kRelayDelay = 4;   // intervals from a chunk's way to LDS to its outputs
constexpr int kRelayHelperThreads = kRelayHelpers * kBlock, kRelayThreads = kRelayHelperThreads + kBlock;
constexpr uint32_t kRelayPadded = 0x7fc0deadu;   // a NaN that no sum of the kernel's own is let be

// Workgroup barrier that orders LDS only: global loads and stores stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// N dwords of LDS, in the widest reads that their place allows
template <int N> __device__ __forceinline__ void lds_words(const char *at, uint32_t (&out)[N]) {
    if constexpr (N % 4 == 0) {
#pragma unroll
        for (int i = 0; i < N / 4; ++i) {
            const u32x4_t v = reinterpret_cast<const u32x4_alias *>(at)[i];
#pragma unroll
            for (int k = 0; k < 4; ++k) out[4 * i + k] = v[k];
        }
    } else if constexpr (N % 2 == 0) {
#pragma unroll
        for (int i = 0; i < N / 2; ++i) {
            const u32x2_t v = reinterpret_cast<const u32x2_alias *>(at)[i];
            out[2 * i] = v[0];
            out[2 * i + 1] = v[1];
        }
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) out[i] = reinterpret_cast<const u32_alias *>(at)[i];
    }
}
// element k of consecutive elements held in dwords
template <typename T, int N> __device__ __forceinline__ float relay_element(const uint32_t (&words)[N], int k) {
    if constexpr (sizeof(T) == 4) return __builtin_bit_cast(float, words[k]);
    else return bits_to_float<T>((k & 1) ? words[k / 2] >> 16 : words[k / 2] & 0xffffu);
}

template <typename T, int K, int SKIP, int MODE, int TC, typename TX = T>
__global__ void __launch_bounds__(kRelayThreads) forward_scan_relay(const FwdParams p) {
    static_assert(TC % kCkptInterval == 0, "a chunk is a whole number of checkpoint intervals");
    constexpr bool PAD = (MODE & kHasPad) != 0, TANH = (MODE & kTanh) != 0;
    constexpr int kS = sizeof(T), kX = SKIP == 1 ? sizeof(TX) : 0;
    constexpr int kRowU = kRelayCols * K * kS, kRowX = kRelayCols * kX;
    constexpr int kPiecesU = TC * kRowU / 16, kPieces = kPiecesU + TC * kRowX / 16;
    constexpr int kMine = (kPieces + kRelayHelperThreads - 1) / kRelayHelperThreads;   // pieces per helper
    constexpr int kCells = TC * (kRelayCols / 2) / kRelayHelperThreads;                // column pairs x steps per helper
    constexpr int kRowStep = kRelayHelperThreads / (kRelayCols / 2);                   // steps between a helper's pairs
    static_assert(kCells >= 1 && kCells * kRowStep == TC, "every helper has the same number of pairs");
    constexpr int A = kS == 4 ? 2 : 4;   // chunks in flight in registers (as many as 256 registers hold)
    constexpr int D = kRelayDelay;
    static_assert(D % A == 0, "the registers of a chunk are indexed by its number modulo A and modulo D");

    __shared__ u32x4_alias raw[2][kPieces];            // elements as they are in memory: U rows, then x rows
    __shared__ f32x4_alias operands[2][TC][kRelayCols / 2];   // (u0, sum) per column
    __shared__ float states[2][TC + 1][kRelayCols];    // row 0: the state before the chunk
    __shared__ int window[2];
    fetch_params_early(p);

    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kBlock));
    const int64_t col0 = (int64_t)blockIdx.x * kRelayCols;
    const int L = (int)p.L, Dp = p.Dp;
    const int64_t ncols = p.ncols;

    // chunks that are walked: those from the first to the last step that is live in any of the rows
    int j0 = 0, j1 = (L + TC - 1) / TC, hi = L;
    if constexpr (PAD) {
        const int64_t b_first = col0 / Dp, b_last = min(col0 + kRelayCols, ncols) - 1;
        const int nb = (int)(b_last / Dp - b_first) + 1;
        if (nb <= 4) {
            if (threadIdx.x == 0) { window[0] = L; window[1] = 0; }
            __syncthreads();
            int first = L, last = 0;   // live times [first, last)
            for (int t = threadIdx.x; t < L; t += kRelayThreads)
                for (int i = 0; i < nb; ++i)
                    if (p.pad[(int64_t)t * p.B + b_first + i] == 0) { first = min(first, t); last = max(last, t + 1); }
#pragma unroll
            for (int off = kBlock / 2; off > 0; off >>= 1) {
                first = min(first, __shfl_xor(first, off, kBlock));
                last = max(last, __shfl_xor(last, off, kBlock));
            }
            if (threadIdx.x % kBlock == 0 && first < last) { atomicMin(&window[0], first); atomicMax(&window[1], last); }
            __syncthreads();
            first = window[0];
            last = window[1];
            if (first >= last) {
                j1 = 0;
                hi = 0;
            } else {   // in walk steps; both ways where the columns go both ways
                const int jf = (int)(col0 % Dp), jl = jf + (int)(min(col0 + kRelayCols, ncols) - col0) - 1;
                const bool some_reverse = p.d < Dp && jl >= p.d, some_forward = jf < p.d || jl >= Dp;
                const int lo = some_reverse ? (some_forward ? min(first, L - last) : L - last) : first;
                hi = some_reverse ? (some_forward ? max(last, L - first) : L - first) : last;
                j0 = lo / TC;
                j1 = (hi + TC - 1) / TC;
                hi = min(j1 * TC, L);
            }
        }
    }
    const int n = j1 - j0;

    if (wave == kRelayHelpers) {
        // ------------------------------------------------------------ the chain
        __builtin_amdgcn_s_setprio(3);
        const int lane = threadIdx.x % kBlock;
        const int64_t col = min(col0 + lane, ncols - 1);
        SmallElem<T> ew, e0;
        const bool wc16 = (p.small16 & kSmallWeightC) != 0, init16 = (p.small16 & kSmallInit) != 0;
        ew.fetch(p.wc, col % Dp, wc16);
        if (p.c0) e0.fetch(p.c0, col, init16);
        const float w1 = kS == 2 ? kNegLog2e * ew.get(wc16) : ew.get(wc16);
        float c = p.c0 ? e0.get(init16) : 0.f;
        f32x2_t now[TC], next[TC];
        // chunk j, while the operands of the next one arrive
        auto walk = [&](int j, const f32x2_t (&ops)[TC], f32x2_t (&to)[TC]) __attribute__((always_inline)) {
            float *out = &states[j & 1][0][lane];
            const f32x2_alias *in = reinterpret_cast<const f32x2_alias *>(&operands[(j + 1) & 1][0][0]) + lane;
            out[0] = c;
#pragma unroll
            for (int r = 0; r < TC; ++r) {
                if (r < TC / 2) {
                    to[2 * r] = in[2 * r * kRelayCols];
                    to[2 * r + 1] = in[(2 * r + 1) * kRelayCols];
                }
                const float u0 = ops[r][0], a = ops[r][1];
                const float t = __builtin_fmaf(w1, c, a);
                const float g = kS == 2 ? sigmoid_exp2<T>(t) : sigmoid_exp2<T>(kNegLog2e * t);
                const float cn = __builtin_fmaf(c - u0, g, u0);
                c = PAD && __builtin_bit_cast(uint32_t, a) == kRelayPadded ? c : cn;
                out[(r + 1) * kRelayCols] = c;
                __builtin_amdgcn_sched_barrier(0);   // (else the reads gather behind the last step, and the barrier waits for them)
                if ((r + 1) % kCkptInterval == 0 && p.ckpt && (j0 + j) * TC + r < L && col0 + lane < ncols)
                    __builtin_nontemporal_store(c, p.ckpt + (int64_t)(((j0 + j) * TC + r) / kCkptInterval) * ncols + col);
            }
        };
        // interval i: operands of chunk i - 2 arrive (one past the last: read and not used), chunk i - 3 is walked
        lds_barrier();
        lds_barrier();
#pragma unroll
        for (int r = 0; r < TC; ++r) now[r] = reinterpret_cast<const f32x2_alias *>(&operands[0][r][0])[lane];
        lds_barrier();
        for (int i = 3; i < n + 3; i += 2) {
            walk(i - 3, now, next);
            lds_barrier();
            if (i + 1 >= n + 3) break;
            walk(i - 2, next, now);
            lds_barrier();
        }
        lds_barrier();
        return;
    }

    // ---------------------------------------------------------------- helpers
    const int tid = threadIdx.x;
    const uint32_t stride_u = (uint32_t)ncols * (K * kS), stride_x = (uint32_t)ncols * (kX ? kX : 1);
    const char *from[kMine];
    uint32_t stride[kMine];
    int row[kMine];
    bool back[kMine];
#pragma unroll
    for (int i = 0; i < kMine; ++i) {
        const int q = min(tid + i * kRelayHelperThreads, kPieces - 1);   // (those past the last repeat it)
        const bool in_u = q < kPiecesU;
        const int at = in_u ? q * 16 : (q - kPiecesU) * 16, pitch = in_u ? kRowU : (kRowX ? kRowX : 1);
        row[i] = at / pitch;
        int within = at % pitch;
        const int per = in_u ? K * kS : (kX ? kX : 1);
        if (col0 + within / per >= ncols) within = 0;   // past the last column
        const int64_t col = col0 + within / per;
        back[i] = col % Dp >= p.d;
        stride[i] = in_u ? stride_u : stride_x;
        from[i] = (in_u ? static_cast<const char *>(p.u) + col0 * (K * kS) : static_cast<const char *>(p.x) + col0 * kX) + within;
    }
    u32x4_t stage[A][kMine];
    auto load = [&](int j, u32x4_t (&to)[kMine]) __attribute__((always_inline)) {   // j: chunk of those that are walked
#pragma unroll
        for (int i = 0; i < kMine; ++i) {
            const int s = min((j0 + j) * TC + row[i], L - 1);
            const uint32_t t = (uint32_t)(back[i] ? L - 1 - s : s);
            to[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t *>(from[i] + (uint64_t)t * stride[i]));
        }
    };

    // this helper's column pair and steps r0, r0 + kRowStep, ... of a chunk
    // (pairs past the last column repeat the last pair in everything they do)
    const int pair = min(tid % (kRelayCols / 2), (int)(min(ncols - col0, (int64_t)kRelayCols) / 2) - 1), r0 = tid / (kRelayCols / 2);
    const int64_t colp = col0 + 2 * pair;
    const int jp = (int)(colp % Dp);
    const int64_t b = colp / Dp;
    const bool rev = jp >= p.d;
    float w2[2], b1[2], b2[2], m[2], init[2], sx = 1.f;
    {
        ColumnOperands<T, 2> op;
        op.fetch(p, p.c0, (p.small16 & kSmallInit) != 0, true, SKIP == 1, jp, colp);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            w2[c] = kS == 2 ? kNegLog2e * op.w2[c] : op.w2[c];
            b1[c] = kS == 2 ? kNegLog2e * op.b1[c] : op.b1[c];
            b2[c] = kS == 2 ? kNegLog2e * op.b2[c] : op.b2[c];
            m[c] = op.m[c];
            init[c] = op.start[c];
        }
        sx = op.sx;
    }
    char *const h = static_cast<char *>(p.h) + colp * kS;
    const uint32_t stride_h = (uint32_t)ncols * kS;
    auto put_h = [&](int s, float a, float c) __attribute__((always_inline)) {
        char *at = h + (uint64_t)(uint32_t)(rev ? L - 1 - s : s) * stride_h;
        if constexpr (kS == 2) __builtin_nontemporal_store(pack_pair<T>(a, c), reinterpret_cast<uint32_t *>(at));
        else __builtin_nontemporal_store(f32x2_t{a, c}, reinterpret_cast<f32x2_t *>(at));
    };
    auto put_ckpt = [&](int s, f32x2_t v) __attribute__((always_inline)) {
        __builtin_nontemporal_store(v, reinterpret_cast<f32x2_t *>(p.ckpt + (int64_t)(s / kCkptInterval) * ncols + colp));
    };

    if constexpr (PAD) {   // what is not walked
        for (int s = r0; s < j0 * TC; s += kRowStep) put_h(s, 0.f, 0.f);
        for (int s = hi + r0; s < L; s += kRowStep) put_h(s, 0.f, 0.f);
        if (p.ckpt)
            for (int s = kCkptInterval * (r0 + 1) - 1; s < (n ? j0 * TC : L); s += kCkptInterval * kRowStep) put_ckpt(s, f32x2_t{init[0], init[1]});
        if (n == 0 && r0 == 0) {
            put_last<T>(p.c_last, colp, init[0], (p.small16 & kSmallLast) != 0);
            put_last<T>(p.c_last, colp + 1, init[1], (p.small16 & kSmallLast) != 0);
        }
    }

    struct Kept { float u2[2], x[2]; } kept[D][kCells];   // the output gate's operands of the chunks under way
    uint32_t flags[A][kCells], gone[kCells];              // padding of chunks to come; of those under way, a bit each
    auto load_flags = [&](int j, uint32_t (&to)[kCells]) __attribute__((always_inline)) {
        if constexpr (PAD) {
#pragma unroll
            for (int i = 0; i < kCells; ++i) {
                const int s = min((j0 + j) * TC + r0 + i * kRowStep, L - 1);
                to[i] = p.pad[(int64_t)(rev ? L - 1 - s : s) * p.B + b];
            }
        }
    };
    struct Words { uint32_t u[2 * K * kS / 4], x[SKIP == 1 ? 2 * kX / 4 : 1]; };   // a column pair's elements of one step
    auto fetch = [&](int j, Words (&words)[kCells]) __attribute__((always_inline)) {
        const char *const base = reinterpret_cast<const char *>(&raw[j & 1][0]);
#pragma unroll
        for (int i = 0; i < kCells; ++i) {
            const int r = r0 + i * kRowStep;
            lds_words<2 * K * kS / 4>(base + r * kRowU + pair * (2 * K * kS), words[i].u);
            if constexpr (SKIP == 1) lds_words<2 * kX / 4>(base + TC * kRowU + r * kRowX + pair * (2 * kX), words[i].x);
        }
    };
    // operands of chunk j for the chain
    auto prepare = [&](int j, const Words (&words)[kCells], Kept (&keep)[kCells], const uint32_t (&flag)[kCells]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kCells; ++i) {
            float u[2][K], sum[2];
#pragma unroll
            for (int k = 0; k < 2 * K; ++k) u[k / K][k % K] = relay_element<T>(words[i].u, k);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                sum[c] = kS == 2 ? __builtin_fmaf(kNegLog2e, u[c][1], b1[c]) : u[c][1] + b1[c];
                if constexpr (PAD) {
                    const uint32_t bits = __builtin_bit_cast(uint32_t, sum[c]);
                    sum[c] = __builtin_bit_cast(float, flag[i] ? kRelayPadded : bits == kRelayPadded ? bits ^ 1u : bits);
                }
                keep[i].u2[c] = kS == 2 ? __builtin_fmaf(kNegLog2e, u[c][2], b2[c]) : u[c][2];
                if constexpr (SKIP == 1) keep[i].x[c] = relay_element<TX>(words[i].x, c) * sx;
                else keep[i].x[c] = u[c][K - 1];
            }
            operands[j & 1][r0 + i * kRowStep][pair] = f32x4_t{u[0][0], sum[0], u[1][0], sum[1]};
            if constexpr (PAD) gone[i] = gone[i] << 1 | (flag[i] != 0);
        }
    };
    auto fetch_states = [&](int j, f32x2_t (&before)[kCells], f32x2_t (&after)[kCells]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kCells; ++i) {
            const int r = r0 + i * kRowStep;
            before[i] = *reinterpret_cast<const f32x2_alias *>(&states[j & 1][r][2 * pair]);
            after[i] = *reinterpret_cast<const f32x2_alias *>(&states[j & 1][r + 1][2 * pair]);
        }
    };
    // outputs of chunk j; LAST: it may end before its last row, and with the walk's last step
    auto finish = [&](int j, const Kept (&keep)[kCells], const f32x2_t (&before)[kCells], const f32x2_t (&after)[kCells], auto last_chunk) __attribute__((always_inline)) {
        constexpr bool LAST = decltype(last_chunk)::value;
#pragma unroll
        for (int i = 0; i < kCells; ++i) {
            const int r = r0 + i * kRowStep, s = (j0 + j) * TC + r;
            float out[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const float g = kS == 2 ? sigmoid_exp2<T>(__builtin_fmaf(w2[c], before[i][c], keep[i].u2[c]))
                                        : sigmoid_exp2<T>(kNegLog2e * (__builtin_fmaf(w2[c], before[i][c], keep[i].u2[c]) + b2[c]));
                const float val = TANH ? tanh_fast(after[i][c]) : after[i][c];
                if constexpr (SKIP != 0) out[c] = __builtin_fmaf((val - keep[i].x[c]) * m[c], g, keep[i].x[c]);
                else out[c] = val * m[c] * g;
                if constexpr (PAD) out[c] = (gone[i] >> 3 & 1) ? 0.f : out[c];
            }
            if constexpr (!LAST) {
                put_h(s, out[0], out[1]);
            } else if (s < L) {
                put_h(s, out[0], out[1]);
                if (s == hi - 1) {
                    put_last<T>(p.c_last, colp, after[i][0], (p.small16 & kSmallLast) != 0);
                    put_last<T>(p.c_last, colp + 1, after[i][1], (p.small16 & kSmallLast) != 0);
                }
            }
        }
    };
    auto put_raw = [&](int j, const u32x4_t (&v)[kMine]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kMine; ++i) raw[j & 1][min(tid + i * kRelayHelperThreads, kPieces - 1)] = v[i];
    };

    // Interval i: chunk i reaches LDS (and chunk i + A is requested in its place), chunk i - 1 is
    // prepared, chunk i - 4 finished. (Loads past the last chunk repeat the last step.) The body of the
    // loop has no branch: with any, the compiler no longer counts the loads in flight and waits for all of
    // them in every interval (58 ns a step instead of 33).
#pragma unroll
    for (int i = 0; i < kCells; ++i) gone[i] = 0;
#pragma unroll
    for (int i = 0; i < A; ++i) {
        load(i, stage[i]);
        load_flags(i, flags[i]);
    }
    // (the flags of chunk i - 1 are where they were loaded; those of chunk i - 1 + A follow them)
    auto interval = [&](int i, auto slot, auto first, auto with_finish, auto last_chunks) __attribute__((always_inline)) {
        constexpr int k = decltype(slot)::value, a = k % A, before = (k + D - 1) % D;
        constexpr bool kPrepare = !decltype(first)::value, kFinish = decltype(with_finish)::value;
        Words words[kCells];
        f32x2_t old[kCells], now[kCells];
        if constexpr (kPrepare) fetch(i - 1, words);
        if constexpr (kFinish) fetch_states(i - 4, old, now);
        put_raw(i, stage[a]);
        load(i + A, stage[a]);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (kPrepare) {
            prepare(i - 1, words, kept[before], flags[before % A]);
            load_flags(i - 1 + A, flags[before % A]);
        }
        // (bit 3 of the flags: those of chunk i - 1 came last)
        if constexpr (kFinish) finish(i - 4, kept[k], old, now, last_chunks);
        lds_barrier();
    };
    using No = std::false_type;
    using Yes = std::true_type;
    interval(0, Int<0>{}, Yes{}, No{}, No{});
    interval(1, Int<1>{}, No{}, No{}, No{});
    interval(2, Int<2>{}, No{}, No{}, No{});
    interval(3, Int<3>{}, No{}, No{}, No{});
    int i = 4;
    for (; i < n; i += D) {
        interval(i, Int<0>{}, No{}, Yes{}, No{});
        interval(i + 1, Int<1>{}, No{}, Yes{}, No{});
        interval(i + 2, Int<2>{}, No{}, Yes{}, No{});
        interval(i + 3, Int<3>{}, No{}, Yes{}, No{});
    }
    if (i < n + 4) interval(i, Int<0>{}, No{}, Yes{}, Yes{});
    if (i + 1 < n + 4) interval(i + 1, Int<1>{}, No{}, Yes{}, Yes{});
    if (i + 2 < n + 4) interval(i + 2, Int<2>{}, No{}, Yes{}, Yes{});
    if (i + 3 < n + 4) interval(i + 3, Int<3>{}, No{}, Yes{}, Yes{});
    if (PAD && p.ckpt && n != 0 && hi < L) {   // the last state, for what is not walked behind it
        const f32x2_t last = *reinterpret_cast<const f32x2_alias *>(&states[(n - 1) & 1][TC][2 * pair]);
        for (int s = hi + kCkptInterval * (r0 + 1) - 1; s < L; s += kCkptInterval * kRowStep) put_ckpt(s, last);
    }
}

}  // namespace sru_amd

// Backward scan for few columns: a team of wavefronts shares one walk.
//
// What bounds it. With fewer columns than a few wavefronts per SIMD a backward walk took the time that one
// wavefront needs for a step after the other (512 steps of 2048 columns bf16 56 us, 8 MB). But only the chain of
// the state's gradient is serial, and it is linear in that gradient:
//   cur' = (q + cur) * a + e,   q, a, e from the states and the streams of the step alone,
// and the states come back from the checkpoints, chunk by chunk. So each wavefront of a workgroup takes another
// chunk of kCkptInterval steps of the same columns, rebuilds its states, folds its steps into one map
// cur' = A * cur + B, and leaves A and B in LDS; behind one barrier every wavefront folds the maps of the
// chunks before its own (in walk order: those later in time) onto the gradient that came into the round,
// and finishes its chunk from there. A round of W wavefronts is W chunks of the walk, loads of the next
// round's chunk are in flight meanwhile.
// Measured (kernel): 512 steps of 2048 columns bf16 56 -> 24 us, float 73 -> 27; 16384 float columns 75 -> 57
// (5.3 TB/s); 32768 bf16 columns 68 -> 61. What bounds it now: instruction issue of the compute units in use for the
// fewest columns (60-72 vector instructions a step of 64 columns, two wavefronts to a SIMD), memory for the most.
//
// Mapping. One column per lane; 16-bit streams move by lane pairs, as in backward_scan_ckpt. The first round
// takes the chunks that do not fill a round, the ragged chunk among them; all other rounds are full, so that
// their loop is straight-line code with a real prefetch in every place.
//
// A map that is not finite (products of up to eight steps' factors can pass the float range where the
// gradient itself does not) shows in the gradient that leaves the round, for every wavefront alike; such a
// round hands the gradient from wavefront to wavefront instead, step by step.
#pragma once

#include "sru_relay.h"

namespace sru_amd {

constexpr int kTeamMax = 8;   // wavefronts of a team, two to a SIMD: 256 registers each

// A pointer that moves from step to step. Where it differs from lane to lane (UNI false) the steps' addresses
// are kept from being computed side by side: two registers per step and stream, which the kernel does not have.
template <typename E, bool UNI> struct Walker {
    E *at;
    int64_t pitch;   // elements
    __device__ __forceinline__ Walker(E *base, int64_t first, int64_t step) : at(base + first), pitch(step) { hide(); }
    __device__ __forceinline__ void next() {
        at += pitch;
        hide();
    }
    __device__ __forceinline__ void hide() {
        if constexpr (!UNI) asm volatile("" : "+v"(at));
    }
};

template <typename T, int K, int SKIP, int MODE, typename TX = T>
__global__ void __launch_bounds__(kBlock * kTeamMax) backward_scan_team(const BwdParams p) {
    static_assert(sizeof(TX) == sizeof(T) || (sizeof(TX) == 4 && SKIP == 1), "a float x next to 16-bit streams");
    constexpr int TC = kCkptInterval;
    constexpr bool NTL = (MODE & kNtLoad) != 0, NTS = (MODE & kNtStore) != 0;
    constexpr bool HAS_PAD = (MODE & kHasPad) != 0, PAIR = (MODE & kPair) != 0, UNI = (MODE & kUniform) != 0;
    constexpr bool TANH = (MODE & kTanh) != 0;
    using SU = Stream<T, K, 1, PAIR>;   // U, grad_u: K elements per column
    using S1 = Stream<T, 1, 1, PAIR>;   // grad_h: one element per column
    using SX = Stream<TX, 1, 1, PAIR && sizeof(TX) == 2>;   // x, grad_x
    __shared__ f32x2_alias maps[2][kTeamMax][kBlock];    // (A, B) of each wavefront's chunk, by the round's parity
    __shared__ float handed[kBlock];
    fetch_params_early(p);

    const int W = (int)(blockDim.x / kBlock);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kBlock));
    const int wlane = (int)(threadIdx.x % kBlock);
    const int q = PAIR ? (wlane & 1) : 0;
    // This lane's column. A workgroup takes up to 64 columns of one direction of one batch row where that wastes few
    // lanes (UNI), else any 64 adjacent columns. Lanes past the last column repeat the last lane, or lane pair, in
    // everything they do.
    int64_t colu, col;
    if constexpr (UNI) {
        const uint32_t per_row = (uint32_t)(p.d + kBlock - 1) / kBlock;
        const uint32_t row = blockIdx.x / per_row, first = (blockIdx.x - row * per_row) * kBlock;
        const int last = PAIR ? (int)(p.d - first) - 2 + q : (int)(p.d - first) - 1;
        colu = (int64_t)row * p.d + first;
        col = colu + (wlane < last ? wlane : last);
    } else {
        const int64_t mine = (int64_t)blockIdx.x * kBlock + wlane, last = PAIR ? p.ncols - 2 + q : p.ncols - 1;
        col = colu = mine < last ? mine : last;
    }
    const uint32_t lane = (uint32_t)(col - colu);
    const int Dp = p.Dp;
    const int ju = (int)(colu % Dp);
    const bool flip = ju >= p.d;

    ColumnOperands<T, 1> op;
    op.fetch(p, p.glast, (p.small16 & kSmallLast) != 0, true, SKIP == 1, ju + (int)lane, col);
    auto &cur = op.start[0];   // d loss / d state: what comes into the round
    CompensatedSum sw1, sw2, sb1, sb2;

    const int64_t L = p.L;
    const int64_t ef = (flip ? (L - 1) : 0) * p.ncols + colu;   // forward-walk step s is at element ef + s * es
    const int64_t es = flip ? -p.ncols : p.ncols;
    const int64_t pf = (flip ? (L - 1) : 0) * p.B + col / Dp;   // (per lane on purpose, see backward_scan_ckpt)
    const int64_t ps = flip ? -p.B : p.B;
    const T *ubase = static_cast<const T *>(p.u);
    const TX *xbase = static_cast<const TX *>(p.x);
    const T *ghbase = static_cast<const T *>(p.gh);
    T *gubase = static_cast<T *>(p.gu);
    TX *gxbase = static_cast<TX *>(p.gx);

    struct Chunk {
        typename SU::G u[TC];
        typename SX::G x[TC];
        typename S1::G gh[TC];
        uint32_t pad[TC];
        float cstart;   // state before the chunk's first step; of chunk 0 without an initial state: any checkpoint
    };
    // n: steps of the chunk (TC except for the ragged one)
    auto load = [&](Chunk &k, int64_t ch, int n) __attribute__((always_inline)) {
        // (the bases are blended with bit masks, the value is dropped when it is used: see backward_scan_ckpt)
        const uintptr_t use_c0 = (ch == 0 && p.c0) ? ~(uintptr_t)0 : (uintptr_t)0;
        const uintptr_t base = (reinterpret_cast<uintptr_t>(p.c0) & use_c0) |
                               (reinterpret_cast<uintptr_t>(p.ckpt + (ch > 0 ? ch - 1 : 0) * p.ncols) & ~use_c0);
        k.cstart = reinterpret_cast<const float *>(base)[col];
        const int64_t e = ef + ch * TC * es;
        Walker<const T, UNI> u(ubase, e * K, es * K), gh(ghbase, e, es);
        Walker<const TX, UNI> x(SKIP == 1 ? xbase : nullptr, SKIP == 1 ? e : 0, es);
        Walker<const uint8_t, false> pad(p.pad, HAS_PAD ? pf + ch * TC * ps : 0, ps);
#pragma unroll
        for (int i = 0; i < TC; ++i) {
            if (i < n) {
                k.u[i] = SU::template load<NTL>(u.at, lane, q);
                if (SKIP == 1) k.x[i] = SX::template load<NTL>(x.at, lane, q);
                k.gh[i] = S1::template load<NTL>(gh.at, lane, q);
                if constexpr (HAS_PAD) k.pad[i] = *pad.at;
                u.next();
                gh.next();
                if (SKIP == 1) x.next();
                if (HAS_PAD) pad.next();
            }
        }
    };

    // GUARD: the first round's, where a chunk may have n < TC steps, or none
    auto compute = [&](const Chunk &k, int64_t ch, int n, int parity, auto guard) __attribute__((always_inline)) {
        constexpr bool GUARD = decltype(guard)::value;
        const int64_t e_last = ef + (ch * TC + TC - 1) * es;   // the chunk is left at its first step
        auto dead = [&](int i) __attribute__((always_inline)) { return (HAS_PAD && k.pad[i] != 0) || (GUARD && i >= n); };
        float st[TC + 1], g1[TC], g2[TC], u0s[TC], xs[TC];
        const uint32_t keep = (ch == 0 && !p.c0) ? 0u : ~0u;
        st[0] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, k.cstart) & keep);
#pragma unroll
        for (int i = 0; i < TC; ++i) {
            float uu[K];
            SU::unpack(k.u[i], q, uu);
            const float cp = st[i];
            u0s[i] = uu[0];
            if (SKIP == 2) xs[i] = uu[K - 1];
            g1[i] = gate<T>(uu[1], op.w1[0], cp, op.b1[0]);
            g2[i] = gate<T>(uu[2], op.w2[0], cp, op.b2[0]);
            const float cn = (cp - u0s[i]) * g1[i] + u0s[i];
            st[i + 1] = dead(i) ? cp : cn;
        }
        // what does not wait for the gradient, and the chunk's map
        float gm[TC], gg2s[TC], d1[TC], gskips[TC];
        float A = 1.f, B = 0.f, gw1 = 0.f, gw2 = 0.f, gb1 = 0.f, gb2 = 0.f;
        Walker<TX, UNI> gxs(SKIP == 1 ? gxbase : nullptr, SKIP == 1 ? e_last : 0, -es);
#pragma unroll
        for (int i = TC - 1; i >= 0; --i) {
            float gx[1], xx[1] = {}, ghs[1];
            if (SKIP == 1) SX::unpack(k.x[i], q, xx);
            S1::unpack(k.gh[i], q, ghs);
            const float val = TANH ? tanh_fast(st[i + 1]) : st[i + 1];
            const float dact = TANH ? (1.0f - val * val) : 1.0f;
            const float G1 = g1[i], G2 = g2[i];
            const float xv = (SKIP == 0) ? 0.0f : (SKIP == 1) ? xx[0] * op.sx : xs[i];
            const float gg2 = ghs[0] * (val - xv) * op.m[0] * (G2 * (1.0f - G2));
            const float gskip = ghs[0] * (1.0f - G2 * op.m[0]);
            gg2s[i] = dead(i) ? 0.0f : gg2;
            gskips[i] = dead(i) ? 0.0f : gskip;
            gm[i] = ghs[0] * op.m[0];
            d1[i] = (st[i] - u0s[i]) * (G1 * (1.0f - G1));
            if constexpr (TANH) g2[i] = G2 * dact;
            const float a = d1[i] * op.w1[0] + G1;
            const float b = (gm[i] * g2[i] + B) * a + gg2s[i] * op.w2[0];
            B = dead(i) ? B : b;
            A = dead(i) ? A : A * a;
            gb2 += gg2s[i];
            gw2 += dead(i) ? 0.0f : gg2s[i] * st[i];
            gx[0] = dead(i) ? 0.0f : gskip * op.sx;
            if constexpr (SKIP == 1) {
                if (!GUARD || i < n) SX::template store<NTS>(gxs.at, lane, q, gx);
                gxs.next();
            }
        }
        // one step of the gradient's chain
        auto back = [&](int i, float from, float &gc, float &gg1) __attribute__((always_inline)) {
            gc = gm[i] * g2[i] + from;
            gg1 = gc * d1[i];
            const float to = gc * g1[i] + gg1 * op.w1[0] + gg2s[i] * op.w2[0];
            return dead(i) ? from : to;
        };
        maps[parity][wave][wlane] = f32x2_t{A, B};
        lds_barrier();
        float mine = cur, carry = cur;   // the gradient that comes into this wavefront's chunk, and out of the round
#pragma unroll
        for (int v = 0; v < kTeamMax; ++v) {
            const f32x2_t f = maps[parity][v][wlane];   // (of wavefronts that are not there: the identity)
            if (v == wave) mine = carry;
            carry = f[0] * carry + f[1];
        }
        const bool finite = __builtin_fabsf(carry) < __builtin_inff();
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(!finite) != 0, 0)) {   // (every wavefront decides from the same numbers)
            carry = cur;
            for (int v = 0; v < W; ++v) {
                if (v == wave) {
                    mine = carry;
                    float run = carry, gc, gg1;
#pragma unroll
                    for (int i = TC - 1; i >= 0; --i) run = back(i, run, gc, gg1);
                    handed[wlane] = run;
                }
                lds_barrier();
                carry = handed[wlane];
                lds_barrier();
            }
        }
        cur = carry;
        Walker<T, UNI> gus(gubase, e_last * K, -es * K);
#pragma unroll
        for (int i = TC - 1; i >= 0; --i) {
            float gu[K], gc, gg1;
            mine = back(i, mine, gc, gg1);
            const float gg1s = dead(i) ? 0.0f : gg1;
            gu[0] = dead(i) ? 0.0f : gc * (1.0f - g1[i]);
            gu[1] = gg1s;
            gu[2] = gg2s[i];
            if (K == 4) gu[K - 1] = gskips[i];
            gb1 += gg1s;
            gw1 += dead(i) ? 0.0f : gg1 * st[i];
            if (!GUARD || i < n) SU::template store<NTS>(gus.at, lane, q, gu);
            gus.next();
        }
        sw1.add(gw1);
        sw2.add(gw2);
        sb1.add(gb1);
        sb2.add(gb2);
    };
    // steps that the window leaves out are known to be padded: no loads, zero gradients
    auto fill = [&](int64_t from, int64_t to) __attribute__((always_inline)) {
        const float zu[K] = {}, z1[1] = {};
        for (int64_t s = from + wave; s < to; s += W) {
            const int64_t e = ef + s * es;
            SU::template store<NTS>(gubase + e * K, lane, q, zu);
            if (SKIP == 1) SX::template store<NTS>(gxbase + e, lane, q, z1);
        }
    };

    int64_t first = 0, end = (L + TC - 1) / TC;   // chunks [first, end) are walked, last to first
    if constexpr (HAS_PAD && UNI) {
        const LiveWindow w = live_window(p.pad, pf, ps, L);   // the same for every wavefront of the team
        first = w.lo / TC;
        end = (w.hi + TC - 1) / TC;
        if (end < first) end = first;
        fill(end * TC, L);
        fill(0, first * TC);
    }
    for (int v = W + wave; v < kTeamMax; v += W)
        maps[0][v][wlane] = maps[1][v][wlane] = f32x2_t{1.f, 0.f};

    if (end > first) {
        const int64_t rounds = (end - first + W - 1) / W;
        const int in_first = (int)(end - first - (rounds - 1) * W);   // chunks of the first round
        Chunk ka = {}, kb;
        int64_t ch = end - 1 - wave;                 // this wavefront's chunk of the first round
        const int n0 = wave < in_first ? (int)min((int64_t)TC, L - ch * TC) : 0;
        if (n0 > 0) load(ka, ch, n0);
        int64_t next = end - in_first - 1 - wave;    // ... and of the next one
        if (rounds > 1) load(kb, next, TC);
        compute(ka, n0 > 0 ? ch : 1, n0, 0, std::true_type{});
        int64_t left = rounds - 1;                   // rounds to come; the first of them is in kb
        while (left >= 3) {
            load(ka, next - W, TC);
            compute(kb, next, TC, 1, std::false_type{});
            __builtin_amdgcn_sched_barrier(0);
            load(kb, next - 2 * W, TC);
            compute(ka, next - W, TC, 0, std::false_type{});
            __builtin_amdgcn_sched_barrier(0);
            next -= 2 * W;
            left -= 2;
        }
        if (left == 2) {
            load(ka, next - W, TC);
            compute(kb, next, TC, 1, std::false_type{});
            compute(ka, next - W, TC, 0, std::false_type{});
        } else if (left == 1) {
            compute(kb, next, TC, 1, std::false_type{});
        }
    }

    // the wavefronts' sums, added in their order (column by column by the wavefronts in turn)
    __shared__ float sums[kTeamMax][4][kBlock];
    sums[wave][0][wlane] = sw1.value();
    sums[wave][1][wlane] = sw2.value();
    sums[wave][2][wlane] = sb1.value();
    sums[wave][3][wlane] = sb2.value();
    lds_barrier();
    for (int quantity = wave; quantity < 4; quantity += W) {
        CompensatedSum total;
        for (int v = 0; v < W; ++v) total.add(sums[v][quantity][wlane]);
        p.partial[quantity * p.ncols + col] = total.value();
    }
    if (wave == 0) p.ginit[col] = cur;
}

}  // namespace sru_amd

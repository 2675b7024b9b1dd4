// Kernel selection for one stream element type T. Included by scan_<type>_fwd.hip, scan_<type>_bwd.hip and
// scan_f64.hip only.
//
// Fast kernels exist for the three layouts the SRU layer produces without a per-step
// weight_c: (k=3, skip from x), (k=3, no skip term) and (k=4, skip from U[..., 3]); whether a
// padding mask is given, whether and how c is stored and the activation are compiled in.
// Everything else (per-step weight_c; k=4 without a skip term, which the layer never
// produces) runs the general kernels, one column per lane. Double streams run the general
// kernels for everything, computing in double.
//
// Every launcher returns the status of its own hipLaunchKernel call; nothing here reads or
// clears the runtime's sticky error state, which may hold an error of the embedding program.
#pragma once

#include <algorithm>

#include "sru_launch.h"
#include "sru_relay.h"
#include "sru_split.h"
#include "sru_team.h"

namespace sru_amd {

// Columns per lane of the fast kernels, per element type: float streams move as dwordx3 /
// dwordx4 per column already; 16-bit streams need two columns per lane (or paired lanes)
// for dword-granular accesses.
template <typename T> struct Tune { static constexpr int kCols = sizeof(T) == 2 ? 2 : 1; };
constexpr int kRingDepth = 8;  // ring kernels (reference-style state, general modes)
// (double streams: a slot is twice as wide, so half the slots keep the ring in registers)
template <typename T> constexpr int general_ring_depth() { return sizeof(T) == 8 ? kRingDepth / 2 : kRingDepth; }
// Every large stream is touched exactly once per kernel, so loads and stores are marked
// non-temporal: measured at the headline shape with cache-cold operands, forward + backward
// 447 us -> 425 us (float), 230 us -> 214 us (bfloat16).
constexpr int kNt = kNtLoad | kNtStore;
// 16-bit streams with few columns: below this many lanes at two columns per lane (fewer than
// 1024 wavefronts) the kernels keep one column per lane and pair lanes for memory access.
#ifndef SRU_AMD_PAIR_BELOW   // (set by tuning builds only)
#define SRU_AMD_PAIR_BELOW 65536
#endif
constexpr int64_t kPairBelow = SRU_AMD_PAIR_BELOW;

// Lane-pair kernels (sru_split.h): 16-bit streams, d a multiple of 32, at most 1024 wavefronts of 32
// columns, every stream 16-byte aligned, state kept as checkpoints or not at all.
#ifndef SRU_AMD_SPLIT_NBUF   // (set by tuning builds only)
#define SRU_AMD_SPLIT_NBUF 2
#endif
constexpr int kSplitNbuf = SRU_AMD_SPLIT_NBUF;   // chunks (of 16 steps) in flight per wavefront
#ifndef SRU_AMD_SPLIT_MAX_WAVES   // (set by tuning builds only)
#define SRU_AMD_SPLIT_MAX_WAVES 1024
#endif
inline bool split_wanted(int64_t ncols, int32_t d) { return d % kSplitCols == 0 && ncols / kSplitCols <= SRU_AMD_SPLIT_MAX_WAVES; }

inline bool aligned_to(const void *p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

// launch of a lane-pair kernel: wavefronts of 32 columns, kSplitWaves per workgroup
template <typename P>
inline hipError_t launch_split(void (*kernel)(P), hipStream_t st, const P &p) {
    void *args[] = {const_cast<P *>(&p)};
    const int64_t wavefronts = p.ncols / kSplitCols;
    return hipLaunchKernel(reinterpret_cast<const void *>(kernel), dim3((unsigned)((wavefronts + kSplitWaves - 1) / kSplitWaves)),
                           dim3(kBlock * kSplitWaves), args, 0, st);
}

// Wavefronts per workgroup for the chunked kernels: 8 or 4 (as the kernel allows) while the launch
// still has a workgroup for each of the 256 compute units, else 1. (Not 2: workgroups of two
// wavefronts measured up to 25 % slower than either neighbour.)
inline int waves_per_group(int64_t wavefronts, int most) {
    for (int n = most; n >= 4; n /= 2)
        if (wavefronts / n >= 256) return n;
    return 1;
}
// launch of a chunked kernel: `most` wavefronts per workgroup at most
template <typename P>
inline hipError_t launch_grouped(void (*kernel)(P), int64_t ncols, int cols, int most, hipStream_t st, const P &p) {
    const int64_t wavefronts = (ncols / cols + kBlock - 1) / kBlock;
    const int n = waves_per_group(wavefronts, most);
    void *args[] = {const_cast<P *>(&p)};
    return hipLaunchKernel(reinterpret_cast<const void *>(kernel), dim3((unsigned)((wavefronts + n - 1) / n)), dim3(kBlock * n),
                           args, 0, st);
}

// Two columns per lane need an even d (a pair must not straddle a direction or a batch
// row) and stream pointers aligned to the pair groups.
template <typename T, int K>
bool pair_ok(const sru_amd_shape &s, std::initializer_list<const void *> wide,
             std::initializer_list<const void *> narrow) {
    if (Tune<T>::kCols != 2 || (s.hidden % 2) != 0) return false;
    const size_t es = sizeof(T);
    for (const void *q : wide)
        if (q && !aligned_to(q, group_align((int)(2 * K * es)))) return false;
    for (const void *q : narrow)
        if (q && !aligned_to(q, group_align((int)(2 * es)))) return false;
    return true;
}

// true when every wavefront lies inside one direction and one batch row
inline bool wave_uniform(int32_t d, int cols) { return d % (kBlock * cols) == 0; }

// X: the template bits fixed so far (pairing, then uniformity, then activation); the run-time
// properties are turned into template bits one at a time.
// TX: element type of x / grad_x (T, or float next to 16-bit streams: those builds exist for the
// identity activation, checkpointed or no state, no per-step weight_c; callers start them at STAGE 1).
template <typename T, int K, int SKIP, int COLS, int X = 0, int STAGE = 0, typename TX = T>
hipError_t fast_forward(const FwdParams &p, hipStream_t st) {
    if constexpr (STAGE == 0 && (X & kCustom) != 0) {   // (a per-step weight_c with tanh runs the general kernels)
        return fast_forward<T, K, SKIP, COLS, X, 1, TX>(p, st);
    } else if constexpr (STAGE == 0) {
        return p.act ? fast_forward<T, K, SKIP, COLS, X | kTanh, 1, TX>(p, st) : fast_forward<T, K, SKIP, COLS, X, 1, TX>(p, st);
    } else if constexpr (STAGE == 1) {
        return wave_uniform(p.d, COLS) ? fast_forward<T, K, SKIP, COLS, X | kUniform, 2, TX>(p, st)
                                       : fast_forward<T, K, SKIP, COLS, X, 2, TX>(p, st);
    } else if constexpr (STAGE == 2) {
        return p.pad ? fast_forward<T, K, SKIP, COLS, X | kHasPad, 3, TX>(p, st) : fast_forward<T, K, SKIP, COLS, X, 3, TX>(p, st);
    } else {
        constexpr int TC = kCkptInterval;
        const int most = max_waves_per_group<T>(X);
        // what is kept for the backward pass: checkpoints, the state after every step, or nothing
        if (p.ckpt) return launch_grouped(forward_scan_chunked<T, K, SKIP, X | kNt | kCkpt, COLS, TC, TX>, p.ncols, COLS, most, st, p);
        // (with a per-step weight_c the state after every step is the general kernels'; with a float x
        // next to 16-bit streams it is refused before)
        if constexpr ((X & kCustom) == 0 && sizeof(TX) == sizeof(T)) {
            if (p.c) return launch_grouped(forward_scan_chunked<T, K, SKIP, X | kNt | kKeepC, COLS, TC>, p.ncols, COLS, most, st, p);
        }
        return launch_grouped(forward_scan_chunked<T, K, SKIP, X | kNt, COLS, TC, TX>, p.ncols, COLS, most, st, p);
    }
}

template <typename T, int K, int SKIP, int COLS, int X = 0, int STAGE = 0, typename TX = T>
hipError_t fast_backward(const BwdParams &p, hipStream_t st) {
    if constexpr (STAGE == 0 && (X & kCustom) != 0) {
        return fast_backward<T, K, SKIP, COLS, X, 1, TX>(p, st);
    } else if constexpr (STAGE == 0) {
        return p.act ? fast_backward<T, K, SKIP, COLS, X | kTanh, 1, TX>(p, st) : fast_backward<T, K, SKIP, COLS, X, 1, TX>(p, st);
    } else if constexpr (STAGE == 1) {
        return p.pad ? fast_backward<T, K, SKIP, COLS, X | kHasPad, 2, TX>(p, st) : fast_backward<T, K, SKIP, COLS, X, 2, TX>(p, st);
    } else {
        if constexpr ((X & (kPair | kCustom)) == 0 && sizeof(TX) == sizeof(T)) {   // (lane pairing, the weight_c stream and a float x exist in the chunked kernels only)
            // reference-style state: the ring kernel reads it step by step
            if (!p.ckpt) return launch_grouped(backward_scan<T, K, SKIP, X | kNt, COLS, kRingDepth>, p.ncols, COLS, 4, st, p);
        }
        constexpr int TC = kCkptInterval;
        const int most = max_waves_per_group<T>(X);
        if (wave_uniform(p.d, COLS))
            return launch_grouped(backward_scan_ckpt<T, K, SKIP, X | kNt | kUniform, COLS, TC, TX>, p.ncols, COLS, most, st, p);
        return launch_grouped(backward_scan_ckpt<T, K, SKIP, X | kNt, COLS, TC, TX>, p.ncols, COLS, most, st, p);
    }
}

template <typename T, int K, int SKIP, int X = 0, int STAGE = 0>
hipError_t split_forward(const FwdParams &p, hipStream_t st) {
    if constexpr (STAGE == 0) {
        return p.act ? split_forward<T, K, SKIP, X | kTanh, 1>(p, st) : split_forward<T, K, SKIP, X, 1>(p, st);
    } else if constexpr (STAGE == 1) {
        return p.pad ? split_forward<T, K, SKIP, X | kHasPad, 2>(p, st) : split_forward<T, K, SKIP, X, 2>(p, st);
    } else {
        if (p.ckpt) return launch_split(forward_scan_split<T, K, SKIP, X | kNt | kCkpt, kSplitNbuf>, st, p);
        return launch_split(forward_scan_split<T, K, SKIP, X | kNt, kSplitNbuf>, st, p);
    }
}

template <typename T, int K, int SKIP, int X = 0, int STAGE = 0>
hipError_t split_backward(const BwdParams &p, hipStream_t st) {
    if constexpr (STAGE == 0) {
        return p.act ? split_backward<T, K, SKIP, X | kTanh, 1>(p, st) : split_backward<T, K, SKIP, X, 1>(p, st);
    } else {
        if (p.pad) return launch_split(backward_scan_split<T, K, SKIP, X | kNt | kHasPad, kSplitNbuf>, st, p);
        return launch_split(backward_scan_split<T, K, SKIP, X | kNt, kSplitNbuf>, st, p);
    }
}

inline bool all_aligned_16(std::initializer_list<const void *> ptrs) {
    for (const void *q : ptrs)
        if (q && !aligned_to(q, 16)) return false;
    return true;
}

// Relay kernel (sru_relay.h): few columns, long enough a walk; whole 16-byte pieces of every stream lie in one
// direction and batch row; the state is kept as checkpoints or not at all.
// A workgroup of five wavefronts takes two register files' worth of a SIMD, so a compute unit holds one at a
// time: beyond 256 workgroups (16384 columns) they follow each other (256 steps of 24576 columns bf16: 26.5 us,
// lane pairs 20.7). The walk passes through five stages, 1-2.5 us more than the other kernels need to start.
// Measured (us, the other kernel / this one; k = 3, two directions):
//   bf16, 2048 columns     48 steps 5.6/5.5   96 8.7/7.6    192 14.8/10.9    padded: 48 6.0/7.5   96 9.6/8.8
//   bf16, 16384 columns    48 steps 6.7/6.4   96 9.7/8.5    192 15.6/12.1    padded: 96 10.7/10.7 192 17.3/15.1
//   bf16, d = 152          48 steps 7.5/6.2   96 11.8/8.2   192 20.4/11.9    padded: 48 8.3/8.4   96 13.2/10.6
//   f32, 2048 columns      96 steps 9.5/9.1   192 16.5/13.6                  padded: 96 9.7/9.6   192 17.0/14.0
//   f32, 16384 columns     96 steps 10.2/11.1 192 17.9/15.9                  padded: 96 11.9/12.9 192 20.0/18.1
constexpr int64_t kRelayMaxColumns = 256 * kRelayCols;
template <typename T> inline bool relay_wanted(const FwdParams &p) {
    const int64_t least = (sizeof(T) == 4 ? 128 : 64) + (p.pad ? 40 : 0);
    return !p.c && p.ncols <= kRelayMaxColumns && p.L >= least && p.L < (1 << 30) && p.d % (16 / (int)sizeof(T)) == 0 &&
           all_aligned_16({p.u, p.x}) && aligned_to(p.h, 8) && aligned_to(p.ckpt, 8);
}
template <typename T, int K, int SKIP, typename TX = T, int X = 0, int STAGE = 0>
hipError_t relay_forward(const FwdParams &p, hipStream_t st) {
    if constexpr (STAGE == 0) {
        return p.act ? relay_forward<T, K, SKIP, TX, X | kTanh, 1>(p, st) : relay_forward<T, K, SKIP, TX, X, 1>(p, st);
    } else if constexpr (STAGE == 1) {
        return p.pad ? relay_forward<T, K, SKIP, TX, X | kHasPad, 2>(p, st) : relay_forward<T, K, SKIP, TX, X, 2>(p, st);
    } else {
        void *args[] = {const_cast<FwdParams *>(&p)};
        return hipLaunchKernel(reinterpret_cast<const void *>(forward_scan_relay<T, K, SKIP, X, kRelaySteps, TX>),
                               dim3((unsigned)((p.ncols + kRelayCols - 1) / kRelayCols)), dim3(kRelayThreads), args, 0, st);
    }
}

// Team kernel (sru_team.h): wavefronts of a workgroup share the walk of 64 columns. A workgroup keeps to one
// direction of one batch row where at most a fifth of its lanes is left over: addresses and flags are scalar then,
// and padding at the ends is not walked.
// Eight wavefronts up to 128 workgroups, from the fifth chunk on; else four, up to where the kernels it stands before
// are faster: those gain from more columns, while two of this one's wavefronts to a SIMD are 512 workgroups. Widths that
// are not a multiple of 64 leave lanes over and split cache lines between workgroups, which memory minds the most: in long
// walks without padding, and with a float x (not where the width is a multiple of 32: others there too are the slower
// ones). A walk of few steps past its second chunk costs this kernel a whole chunk.
// Measured (us, backward call with its 4 us reduction, the other kernels / this one; k = 3 and one direction if not said):
//   bf16, d = 512   17 steps   8192 columns 9.3/7.6    32768 10.5/9.2    40960 10.0/12.3
//                   64 steps   8192 13.4/9.2    32768 15.7/13.7   40960 19.3/18.5 (no skip term, padded 18.3/19.0)
//                   96 steps   40960 25.8/23.7 (no skip term, padded 24.0/23.9)   49152 26.0/25.9 (k = 4 23.2/24.9)
//                   256 steps  2048 33.4/18.0  32768 39.6/35.6   40960 55.3/49.5   49152 56.1/53.1 (k = 4, 128 steps 28.8/30.7)
//   with a float x  256 steps  8192 44.1/17.9  32768 47.8/38.8   40960 48.1/52.9
//   bf16, 400 steps d = 1000   25000 columns 80.9/70.8, 32000 78.1/85.8; padded, tanh, k = 4 84.1/60.0; float x 32000 67.9/92.2
//                   d = 250    20000 columns with a float x 0.93 of the others' rate (d = 1014, 52 steps 18432 columns 16.4/13.9)
//                   d = 96     20480 columns 0.93 of the others' rate; with a float x 32768 71.8/63.7
//   bf16, 17 steps  d = 304    24320 columns padded, tanh, k = 4 10.3/10.7
//   f32, d = 512    17 steps 16384 columns 7.9/7.8   64 steps 14.6/11.4   512 steps 77.9/55.1 (padded 96.0/60.9)
//   f32, d = 250    17 steps 16000 columns 8.4/8.9   24 steps 9.0/9.3   64 steps 15.3/13.5   400 steps 61.5/64.5 (12000 61.0/47.9)
inline bool team_by_row(int32_t d) { return (d + kBlock - 1) / kBlock * kBlock * 4 <= d * 5; }
inline int64_t team_groups(int64_t ncols, int32_t d) {
    return team_by_row(d) ? ncols / d * ((d + kBlock - 1) / kBlock) : (ncols + kBlock - 1) / kBlock;
}
inline int team_waves(const BwdParams &p, bool narrow) {   // narrow: 16-bit streams
    const int64_t groups = team_groups(p.ncols, p.d), chunks = (p.L + kCkptInterval - 1) / kCkptInterval;
    const bool whole = p.d % kBlock == 0, rows32 = p.d % 32 == 0;
    if (p.L < (narrow || whole ? 17 : 18)) return 1;
    int64_t most;
    if (!narrow) most = whole || p.pad || p.L < 256 ? 256 : 224;
    else if (whole) most = p.x_float || p.L <= 88 ? 512 : 640;
    else if (p.L < 20) most = 256;
    else if (p.x_float) most = rows32 ? 512 : 288;
    else most = p.pad || p.L < (rows32 ? 64 : 128) ? 512 : rows32 ? 256 : 384;
    if (groups > most) return 1;
    return groups <= 128 && chunks > 4 ? 8 : 4;
}
// X, STAGE, TX: as in fast_forward
template <typename T, int K, int SKIP, int X = 0, int STAGE = 0, typename TX = T>
hipError_t team_backward(const BwdParams &p, int waves, hipStream_t st) {
    if constexpr (STAGE == 0) {
        return p.act ? team_backward<T, K, SKIP, X | kTanh, 1, TX>(p, waves, st) : team_backward<T, K, SKIP, X, 1, TX>(p, waves, st);
    } else if constexpr (STAGE == 1) {
        return p.pad ? team_backward<T, K, SKIP, X | kHasPad, 2, TX>(p, waves, st) : team_backward<T, K, SKIP, X, 2, TX>(p, waves, st);
    } else if constexpr (STAGE == 2) {
        return team_by_row(p.d) ? team_backward<T, K, SKIP, X | kUniform, 3, TX>(p, waves, st)
                                : team_backward<T, K, SKIP, X, 3, TX>(p, waves, st);
    } else {
        void *args[] = {const_cast<BwdParams *>(&p)};
        constexpr int kLanes = sizeof(T) == 2 ? kPair : 0;
        return hipLaunchKernel(reinterpret_cast<const void *>(backward_scan_team<T, K, SKIP, X | kLanes | kNt, TX>),
                               dim3((unsigned)team_groups(p.ncols, p.d)), dim3((unsigned)(kBlock * waves)), args, 0, st);
    }
}

template <typename T, int K, int SKIP>
hipError_t general_forward(const FwdParams &p, hipStream_t st) {
    return launch_grouped(forward_scan<T, K, SKIP, kGeneral | kNt, 1, general_ring_depth<T>()>, p.ncols, 1, 4, st, p);
}
template <typename T, int K, int SKIP>
hipError_t general_backward(const BwdParams &p, hipStream_t st) {
    return launch_grouped(backward_scan<T, K, SKIP, kGeneral | kNt, 1, general_ring_depth<T>()>, p.ncols, 1, 4, st, p);
}

// 16-bit streams whose columns cannot be paired (odd d, or a stream pointer that is not aligned to a
// pair's group) run the general kernels, one column per lane with 2-byte accesses; the host side
// refuses checkpointed state for them.
template <typename T, int K, int SKIP>
hipError_t pick_forward(const sru_amd_shape &s, const FwdParams &p, hipStream_t st) {
    if (!p.x_float && relay_wanted<T>(p)) return relay_forward<T, K, SKIP>(p, st);
    if constexpr (sizeof(T) == 2) {
        if constexpr (SKIP == 1) {
            if (p.x_float) {   // a float x next to 16-bit streams: chunked kernels only (the flag combinations were checked before)
                if (p.act || p.c || !pair_ok<T, K>(s, {p.u}, {p.h}) || !aligned_to(p.x, 4)) return hipErrorInvalidValue;
                if (relay_wanted<T>(p)) return relay_forward<T, K, SKIP, float, 0, 1>(p, st);
                if (p.ncols / 2 < kPairBelow) return fast_forward<T, K, SKIP, 1, kPair, 1, float>(p, st);
                return fast_forward<T, K, SKIP, 2, 0, 1, float>(p, st);
            }
        }
        if (!p.c && split_wanted(p.ncols, p.d) && all_aligned_16({p.u, p.x, p.h}))
            return split_forward<T, K, SKIP>(p, st);
        if (!pair_ok<T, K>(s, {p.u}, {p.x, p.h, p.c}))
            return p.ckpt ? hipErrorInvalidValue : general_forward<T, K, SKIP>(p, st);
        if (p.ncols / 2 < kPairBelow) return fast_forward<T, K, SKIP, 1, kPair>(p, st);
        return fast_forward<T, K, SKIP, 2>(p, st);
    } else {
        return fast_forward<T, K, SKIP, 1>(p, st);
    }
}

template <typename T, int K, int SKIP>
hipError_t pick_backward(const sru_amd_shape &s, const BwdParams &p, hipStream_t st) {
    if constexpr (sizeof(T) == 2) {
        if constexpr (SKIP == 1) {
            if (p.x_float) {
                if (p.act || !p.ckpt || !pair_ok<T, K>(s, {p.u, p.gu}, {p.gh}) || !aligned_to(p.x, 4) || !aligned_to(p.gx, 4))
                    return hipErrorInvalidValue;
                if (const int w = team_waves(p, sizeof(T) == 2); w > 1) return team_backward<T, K, SKIP, 0, 1, float>(p, w, st);
                if (p.ncols / 2 < kPairBelow) return fast_backward<T, K, SKIP, 1, kPair, 1, float>(p, st);
                return fast_backward<T, K, SKIP, 2, 0, 1, float>(p, st);
            }
        }
        if (p.ckpt && pair_ok<T, K>(s, {p.u, p.gu}, {p.x, p.c, p.gh, p.gx}))
            if (const int w = team_waves(p, sizeof(T) == 2); w > 1) return team_backward<T, K, SKIP>(p, w, st);
        if (p.ckpt && split_wanted(p.ncols, p.d) && all_aligned_16({p.u, p.x, p.gh, p.gu, p.gx}))
            return split_backward<T, K, SKIP>(p, st);
        if (!pair_ok<T, K>(s, {p.u, p.gu}, {p.x, p.c, p.gh, p.gx}))   // p.c is null with checkpoints
            return p.ckpt ? hipErrorInvalidValue : general_backward<T, K, SKIP>(p, st);
        if (p.ckpt && p.ncols / 2 < kPairBelow) return fast_backward<T, K, SKIP, 1, kPair>(p, st);
        return fast_backward<T, K, SKIP, 2>(p, st);
    } else {
        if (p.ckpt)
            if (const int w = team_waves(p, sizeof(T) == 2); w > 1) return team_backward<T, K, SKIP>(p, w, st);
        return fast_backward<T, K, SKIP, 1>(p, st);
    }
}

// (k, skip_type) pairs that pass the shape check: (3,0) (3,1) (4,0) (4,2).
// A per-step weight_c runs the chunked kernels (with the weight_c stream compiled in) when the
// activation is the identity, the state is kept as checkpoints or not at all, and, for 16-bit
// streams, columns can be paired; everything else about it is the general kernels' business.
template <typename T, int K>
bool custom_chunked_ok(const sru_amd_shape &s, bool full_state, std::initializer_list<const void *> wide,
                       std::initializer_list<const void *> mid, std::initializer_list<const void *> narrow) {
    if (!s.is_custom || s.activation_type != 0 || full_state || (s.skip_type == 0 && s.k == 4)) return false;
    if (sizeof(T) == 4) return true;
    for (const void *q : mid)
        if (q && !aligned_to(q, 8)) return false;
    return pair_ok<T, K>(s, wide, narrow);
}

template <typename T, int K, int SKIP>
hipError_t custom_forward(const FwdParams &p, hipStream_t st) {
    return fast_forward<T, K, SKIP, Tune<T>::kCols, kCustom>(p, st);
}
template <typename T, int K, int SKIP>
hipError_t custom_backward(const BwdParams &p, hipStream_t st) {
    return fast_backward<T, K, SKIP, Tune<T>::kCols, kCustom>(p, st);
}

template <typename T>
hipError_t launch_forward(const sru_amd_shape &s, const FwdParams &p, hipStream_t st) {
    if constexpr (sizeof(T) != 8) {
        if (s.k == 3 ? custom_chunked_ok<T, 3>(s, p.c != nullptr, {p.u}, {p.wc}, {p.x, p.h})
                     : custom_chunked_ok<T, 4>(s, p.c != nullptr, {p.u}, {p.wc}, {p.x, p.h})) {
            if (s.k == 4) return custom_forward<T, 4, 2>(p, st);
            if (s.skip_type == 1) return custom_forward<T, 3, 1>(p, st);
            return custom_forward<T, 3, 0>(p, st);
        }
        const bool general = s.is_custom != 0 || (s.skip_type == 0 && s.k == 4);
        if (!general) {
            if (s.k == 4) return pick_forward<T, 4, 2>(s, p, st);
            if (s.skip_type == 1) return pick_forward<T, 3, 1>(s, p, st);
            return pick_forward<T, 3, 0>(s, p, st);
        }
    }
    if (s.k == 3 && s.skip_type == 1) return general_forward<T, 3, 1>(p, st);
    if (s.k == 3) return general_forward<T, 3, 0>(p, st);
    if (s.skip_type == 2) return general_forward<T, 4, 2>(p, st);
    return general_forward<T, 4, 0>(p, st);
}

template <typename T>
hipError_t launch_backward(const sru_amd_shape &s, const BwdParams &p, hipStream_t st) {
    if constexpr (sizeof(T) != 8) {
        if (s.k == 3 ? custom_chunked_ok<T, 3>(s, p.ckpt == nullptr, {p.u, p.gu}, {p.wc, p.gwc_steps}, {p.x, p.gh, p.gx})
                     : custom_chunked_ok<T, 4>(s, p.ckpt == nullptr, {p.u, p.gu}, {p.wc, p.gwc_steps}, {p.x, p.gh, p.gx})) {
            if (s.k == 4) return custom_backward<T, 4, 2>(p, st);
            if (s.skip_type == 1) return custom_backward<T, 3, 1>(p, st);
            return custom_backward<T, 3, 0>(p, st);
        }
        const bool general = s.is_custom != 0 || (s.skip_type == 0 && s.k == 4);
        if (!general) {
            if (s.k == 4) return pick_backward<T, 4, 2>(s, p, st);
            if (s.skip_type == 1) return pick_backward<T, 3, 1>(s, p, st);
            return pick_backward<T, 3, 0>(s, p, st);
        }
    }
    if (p.ckpt) return hipErrorInvalidValue;   // the general kernels read the state after every step (refused by the shape and alignment checks before)
    if (s.k == 3 && s.skip_type == 1) return general_backward<T, 3, 1>(p, st);
    if (s.k == 3) return general_backward<T, 3, 0>(p, st);
    if (s.skip_type == 2) return general_backward<T, 4, 2>(p, st);
    return general_backward<T, 4, 0>(p, st);
}

}  // namespace sru_amd

// Dense product of a layer without gradients, out = x weight, at the sizes where a library product is mostly
// latency: a short sequence, a prompt of one or a few sequences.
//
// What bounds it: latency, of the launch and of the tiles of inner indices that follow each other (2.4 us for an empty
// one, 0.15-0.3 us a tile); at the largest sizes that it takes, LDS and instruction issue. Against the library, us
// in a graph: bf16 512 x 2048 -> 512 10.8 -> 8.8, 512 x 512 -> 6144 12.9 -> 11.3, 128 x 1024 -> 256 10.5 -> 4.8; float
// 640 x 128 -> 384 4.3 -> 3.4, 2048 x 256 -> 768 22.3 -> 12.2. More in sru_layer.h, where the tile is chosen.
//
// Mapping. Four wavefronts own a tile of 32 TM rows by 32 TN columns, each a quarter of it; with G of two such groups
// share the tile and take every other tile of inner indices, and their sums meet in LDS. Inner indices
// come 128 bytes of a row of x at a time; kAhead such tiles are in flight in registers, one is in LDS and one on its
// way there, one barrier a tile. Matrix instructions want consecutive inner indices of a row of x and of a column of
// the weight: x goes to LDS as it is, in pieces of 16 bytes, and of the weight a thread loads the same four bytes
// of four rows and leaves them as one or two columns of four. Addresses are buffer offsets, the tile's part of them
// scalar (64-bit pointers per lane took 5-20% longer). The weight is the first operand of the matrix
// instruction, so that a lane ends with four adjacent columns of a row. Workgroups that share an XCD (every
// eighth) take adjacent tiles of the same columns.
#include "sru_amd.h"

#include <hip/hip_runtime.h>

#include "sru_layer.h"
#include "sru_mfma.h"
#include "sru_relay.h"

namespace sru_amd {
namespace {

constexpr int kQuads = 4;         // wavefronts that share a tile of inner indices
constexpr int kGroupThreads = kQuads * kBlock;
constexpr int kAhead = 4;         // tiles in flight (even: the half of LDS stays static)

// Bytes of memory behind a base that all lanes share.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00027000);
}

template <typename T, int TM, int TN, int G>
__global__ void __launch_bounds__(kGroupThreads * G) product_tile(const ProductParams p) {
    constexpr int ES = sizeof(T), BM = 32 * TM, BN = 32 * TN, BK = 128 / ES;
    constexpr int KP = 16 / ES;                       // inner indices of a 16-byte piece of x
    constexpr int kPitchA = BM + 2;                   // pieces; the padding spreads the writes of a row over the banks
    constexpr int kAtoms = BK / 4;                    // of four inner indices
    constexpr int kPitchB = BN + (ES == 2 ? 8 : 2);   // atoms; 16-bit reads of two rows of atoms meet on different banks
    constexpr int kPerDword = 4 / ES, kUnits = BN / kPerDword;   // columns of a thread's four bytes, such units of a row
    typedef uint32_t atom_t __attribute__((ext_vector_type(ES == 2 ? 2 : 4), may_alias));
    struct Lds {
        u32x4_alias a[2][8 * kPitchA];
        atom_t b[2][kAtoms * kPitchB];
    };
    constexpr int kSums = (G - 1) * TM * TN * kGroupThreads;
    __shared__ __attribute__((aligned(16))) union Shared {
        __device__ Shared() {}
        Lds lds[G];
        f32x4_alias sums[kSums ? kSums : 1];
    } shared;

    const int M = p.rows, N = p.cols, K = p.inner;
    const int tiles_m = (M + BM - 1) / BM, tiles = tiles_m * ((N + BN - 1) / BN), share = (tiles + 7) / 8;
    const int tile = (int)(blockIdx.x % 8) * share + (int)(blockIdx.x / 8);
    if (tile >= tiles) return;
    const int row0 = tile % tiles_m * BM, col0 = tile / tiles_m * BN;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kBlock)), group = wave / kQuads, quad = wave % kQuads;
    const int tid = threadIdx.x % kGroupThreads;
    Lds &lds = shared.lds[group];

    // Tile i of this group starts at inner index first + i * G * BK, so that the last one of all ends with the
    // last inner index and only the first ones have places before inner index 0.
    const int n = ((K + BK - 1) / BK + G - 1) / G, first = K - (n * G - group) * BK;
    const __amdgpu_buffer_rsrc_t xs = buffer(p.x, (uint32_t)M * K * ES), ws = buffer(p.weight, (uint32_t)K * N * ES);
    const int pitch = N * ES;
    // this thread's pieces of x and units of the weight in a tile (rows and columns past the last repeat it and are dropped)
    const int ka = tid % 8 * KP, row_in = tid / 8, kb = tid / kUnits * 4, unit = tid % kUnits;
    constexpr int kRowsA = kGroupThreads / 8, kStepB = kGroupThreads / kUnits * 4;
    int xa[TM], wb[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) xa[i] = (min(row0 + row_in + i * kRowsA, M - 1) * K + ka) * ES;
    const int col_in = min(col0 + unit * kPerDword, N - kPerDword);
#pragma unroll
    for (int i = 0; i < TN; ++i) wb[i] = (kb + i * kStepB) * pitch + col_in * ES;

    struct Stage {
        u32x4 a[TM];
        uint32_t b[TN][4];
    } stage[kAhead];
    auto load = [&](int i, Stage &to) __attribute__((always_inline)) {   // a tile that is all there
        const int k0 = first + i * (G * BK);
#pragma unroll
        for (int j = 0; j < TM; ++j) to.a[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xs, xa[j], k0 * ES, 0));
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) to.b[j][r] = __builtin_amdgcn_raw_buffer_load_b32(ws, wb[j], (k0 + r) * pitch, 0);
    };
    auto load_any = [&](int i, Stage &to) __attribute__((always_inline)) {   // inner indices that are not there repeat others
        const int k0 = first + i * (G * BK);
#pragma unroll
        for (int j = 0; j < TM; ++j)
            to.a[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xs, xa[j] + (min(max(k0 + ka, 0), K - KP) - ka) * ES, 0, 0));
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int at = min(max(k0 + kb + j * kStepB, 0), K - 4) * pitch + col_in * ES;
#pragma unroll
            for (int r = 0; r < 4; ++r) to.b[j][r] = __builtin_amdgcn_raw_buffer_load_b32(ws, at, r * pitch, 0);
        }
    };
    auto put = [&](const Stage &from, int half) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < TM; ++j) lds.a[half][tid % 8 * kPitchA + row_in + j * kRowsA] = from.a[j];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const uint32_t (&b)[4] = from.b[j];
            u32x4 v;
            if constexpr (ES == 2)
                v = u32x4{__builtin_amdgcn_perm(b[1], b[0], 0x05040100u), __builtin_amdgcn_perm(b[3], b[2], 0x05040100u),
                          __builtin_amdgcn_perm(b[1], b[0], 0x07060302u), __builtin_amdgcn_perm(b[3], b[2], 0x07060302u)};
            else
                v = u32x4{b[0], b[1], b[2], b[3]};
            *reinterpret_cast<u32x4_alias *>(&lds.b[half][(kb + j * kStepB) / 4 * kPitchB + unit * kPerDword]) = v;
        }
    };

    const int lane = threadIdx.x % kBlock, m = lane % 16, q = lane / 16;
    const int wave_row = quad / 2 * (BM / 2), wave_col = quad % 2 * (BN / 2);
    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](int half) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {   // four pieces of each row at a time
            u32x4 x[TM], w[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) x[i] = lds.a[half][(4 * s + q) * kPitchA + wave_row + 16 * i + m];
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int col = wave_col + 16 * j + m;
                if constexpr (ES == 2) {
                    const atom_t lo = lds.b[half][(8 * s + 2 * q) * kPitchB + col], hi = lds.b[half][(8 * s + 2 * q + 1) * kPitchB + col];
                    w[j] = u32x4{lo[0], lo[1], hi[0], hi[1]};
                } else {
                    w[j] = lds.b[half][(4 * s + q) * kPitchB + col];
                }
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    if constexpr (ES == 2) {
                        acc[i][j] = mfma<T>(w[j], x[i], acc[i][j]);
                    } else {   // (instruction e multiplies inner indices e, 4 + e, 8 + e and 12 + e)
                        const f32x4 wf = __builtin_bit_cast(f32x4, w[j]), xf = __builtin_bit_cast(f32x4, x[i]);
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[e], xf[e], acc[i][j], 0, 0, 0);
                    }
                }
        }
    };

#pragma unroll
    for (int i = 0; i < kAhead; ++i) load_any(i, stage[i]);
#pragma unroll
    for (int j = 0; j < TM; ++j)
        if (first + ka < 0) stage[0].a[j] = u32x4{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) stage[0].b[j][r] = first + kb + j * kStepB < 0 ? 0u : stage[0].b[j][r];
    // (loads past the last tile repeat it; the loop's body has no branch, so that the compiler counts the loads in
    // flight instead of waiting for all of them)
    int t = 0;
    for (; n - t > kAhead; t += kAhead) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            put(stage[i], i & 1);
            load(min(t + i + kAhead, n - 1), stage[i]);
            lds_barrier();
            multiply(i & 1);
        }
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
        if (t + i < n) {
            put(stage[i], i & 1);
            lds_barrier();
            multiply(i & 1);
        }
    }

    if constexpr (G > 1) {   // the groups' sums, added in their order
        __syncthreads();
        if (group > 0) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) shared.sums[((group - 1) * TM * TN + i * TN + j) * kGroupThreads + tid] = acc[i][j];
        }
        __syncthreads();
        if (group > 0) return;
#pragma unroll
        for (int g = 0; g < G - 1; ++g)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] += shared.sums[(g * TM * TN + i * TN + j) * kGroupThreads + tid];
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int row = row0 + wave_row + 16 * i + m;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int col = col0 + wave_col + 16 * j + 4 * q;
            if (row >= M || col >= N) continue;
            const f32x4 v = acc[i][j];
            if constexpr (ES == 2)
                *reinterpret_cast<u32x2 *>(static_cast<uint16_t *>(p.out) + (int64_t)row * N + col) = u32x2{pack_pair<T>(v[0], v[1]), pack_pair<T>(v[2], v[3])};
            else
                *reinterpret_cast<f32x4 *>(static_cast<float *>(p.out) + (int64_t)row * N + col) = v;
        }
    }
}

template <typename T, int TM, int TN, int G> hipError_t launch(const ProductParams &p, hipStream_t st) {
    const int64_t tiles = (int64_t)((p.rows + 32 * TM - 1) / (32 * TM)) * ((p.cols + 32 * TN - 1) / (32 * TN));
    void *args[] = {const_cast<ProductParams *>(&p)};
    return hipLaunchKernel(reinterpret_cast<const void *>(product_tile<T, TM, TN, G>), dim3((unsigned)((tiles + 7) / 8 * 8)),
                           dim3(kGroupThreads * G), args, 0, st);
}
template <typename T> hipError_t product_of(const ProductParams &p, const ProductTile &t, hipStream_t st) {
    if constexpr (sizeof(T) == 2) {   // (in float larger tiles come with more workgroups than a split wants)
        if (t.split == 2 && t.n == 2) return t.m == 2 ? launch<T, 2, 2, 2>(p, st) : launch<T, 1, 2, 2>(p, st);
    }
    if (t.n == 2) return t.m == 2 ? launch<T, 2, 2, 1>(p, st) : launch<T, 1, 2, 1>(p, st);
    return t.split == 2 ? launch<T, 1, 1, 2>(p, st) : launch<T, 1, 1, 1>(p, st);
}

}  // namespace

hipError_t launch_product(const ProductParams &p, int32_t dtype, const ProductTile &tile, hipStream_t st) {
    if (dtype == SRU_AMD_F32) return product_of<float>(p, tile, st);
    return dtype == SRU_AMD_F16 ? product_of<half_bits>(p, tile, st) : product_of<bf16_bits>(p, tile, st);
}

}  // namespace sru_amd

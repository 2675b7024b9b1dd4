// Weight gradient of a layer's dense product, grad (inner, cols) = x^T g: a contraction over all rows of x (rows, inner)
// and g (rows, cols), of which a small result is left.
//
// What bounds it: the result is small, so the library's tiles of it leave compute units idle or walk all rows one after
// the other (8192 rows, 512 x 6144: 92 us, 560 TFLOP/s; 256 x 1024: 54 us). Here the rows are split as well, in as many
// parts as fill the chip with one round of workgroups (sru_layer.h), float slices of the result meet in a second
// launch, and that launch writes the gradient in the type of the parameter: under autocast in float, which
// takes the library a conversion pass over a gradient rounded to 16 bits.
// A walk that is alone on its compute unit waits for itself: of 0.9 us for a tile of 64 rows its matrix cores were busy
// 0.33, LDS, which every operand passes twice, 0.4, and the loads as much, and they overlapped little. So two teams of
// four wavefronts walk the even and the odd tiles of a part, each with its own two tiles in LDS, and at the end each
// hands the other half of its sums: 0.76 us a tile, 8192 rows, 512 x 6144 71 -> 65 us with the slices' sum, 2048 x 512
// 33.5 -> 30.5, 34393 rows, 504 x 2496 131 -> 108; 67 sizes 0.93 of the time before. The products of a part then take
// place at 1.03 PFLOP/s, and 14 of the 65 us go to the slices. Measured against it: a second tile in flight of a single
// team (level), a workgroup order by which an XCD reads all of g (18% slower), 64-bit addresses per lane; more parts
// instead of teams pay for more slices.
//
// Mapping. A workgroup owns 128 columns of x by 128 or 192 of g, its teams walk their tiles 64 rows at a time: one tile
// is in LDS as it is in memory, the next in registers on its way there, one barrier a tile. Both operands
// want consecutive rows of a column, which the transposing LDS read gives. The columns of g are the first operand of
// the matrix instruction, so that a lane ends with four adjacent ones of a row of the result.
#include "sru_amd.h"

#include <hip/hip_runtime.h>

#include "sru_layer.h"
#include "sru_mfma.h"
#include "sru_relay.h"

namespace sru_amd {
namespace {

constexpr int kGradTeam = 4 * kBlock, kGradThreads = 2 * kGradTeam, kGradRows = 64;   // rows of x and g in a tile
constexpr int kGradTileM = 128;

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 *lds_s16x4;

// c += a b for 32 x 16 times 16 x 32: lane (h, m) = (lane / 32, lane % 32) holds row m of a and column m of b, inner
// indices 8h .. 8h + 7, and of column m of c rows 8i + 4h .. 8i + 4h + 3 in elements 4i .. 4i + 3.
template <typename T> __device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c);
template <> __device__ __forceinline__ f32x16 mfma32<bf16_bits>(u32x4 a, u32x4 b, f32x16 c) {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}
template <> __device__ __forceinline__ f32x16 mfma32<half_bits>(u32x4 a, u32x4 b, f32x16 c) {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}

// Where 16-byte piece c of row r of a tile of W columns stands in its row. Four rows of a column are read together,
// 64 bytes of each, and must meet on different banks.
template <int W> __device__ __forceinline__ int grad_piece(int r, int c) {
    if constexpr (W % 128 == 0) return c ^ ((r & 3) << 2);
    else return c ^ ((r >> 1 & 1) << 2);   // (192 columns: rows two apart start on the same bank)
}

// NT: 32-wide column tiles of a wavefront
template <typename T, int NT>
__global__ void __launch_bounds__(kGradThreads, 2) product_grad(const GradParams p) {
    constexpr int BM = kGradTileM, BN = 64 * NT, CA = BM / 8, CB = BN / 8;   // columns, 16-byte pieces of a row
    constexpr int UA = kGradRows * CA / kGradTeam, UB = kGradRows * CB / kGradTeam;
    constexpr int TA = kGradRows * CA, TB = kGradRows * CB;
    __shared__ u32x4_alias memory[4 * (TA + TB)];   // two tiles of each team

    const int M = p.inner, N = p.cols, R = p.rows;
    const int tiles_m = (M + BM - 1) / BM, tiles = tiles_m * ((N + BN - 1) / BN);
    // workgroups that share an XCD (every eighth) take adjacent tiles of the same rows
    const int share = (tiles * p.splits + 7) / 8, id = (int)(blockIdx.x % 8) * share + (int)(blockIdx.x / 8);
    if (id >= tiles * p.splits) return;
    const int tile = id % tiles, split = id / tiles;
    const int m0 = tile % tiles_m * BM, n0 = tile / tiles_m * BN;
    // Tiles of rows end with the last row, so that only the first one can have places before row 0.
    const int all = (R + kGradRows - 1) / kGradRows;
    const int t0 = (int)((int64_t)all * split / p.splits), n = (int)((int64_t)all * (split + 1) / p.splits) - t0;
    const int first = R - (all - t0) * kGradRows;
    const int team = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kGradTeam), tid = threadIdx.x % kGradTeam;
    u32x4_alias *const as = memory + team * 2 * TA, *const bs = memory + 4 * TA + team * 2 * TB;
    const int mine = (n - team + 1) / 2, most = (n + 1) / 2;   // tiles: the even ones of one team, the odd ones of the other

    // (columns past the last repeat it and are dropped)
    const __amdgpu_buffer_rsrc_t xs = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p.x), 0, (int)((uint32_t)R * M * 2), 0x00027000);
    const __amdgpu_buffer_rsrc_t gs = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p.g), 0, (int)((uint32_t)R * N * 2), 0x00027000);
    int ra[UA], rb[UB], xa[UA], gb[UB], wa[UA], wb[UB];   // row of the tile, byte in memory from its first row, piece in LDS
#pragma unroll
    for (int i = 0; i < UA; ++i) {
        const int id = tid + i * kGradTeam, r = id / CA, c = id % CA;
        ra[i] = r;
        wa[i] = r * CA + grad_piece<BM>(r, c);
        xa[i] = r * M * 2 + min(m0 + c * 8, M - 8) * 2;
    }
#pragma unroll
    for (int i = 0; i < UB; ++i) {
        const int id = tid + i * kGradTeam, r = id / CB, c = id % CB;
        rb[i] = r;
        wb[i] = r * CB + grad_piece<BN>(r, c);
        gb[i] = r * N * 2 + min(n0 + c * 8, N - 8) * 2;
    }
    u32x4 sa[UA], sb[UB];   // the tile on its way from memory to LDS
    auto load = [&](int t) __attribute__((always_inline)) {
        const int r0 = first + (2 * t + team) * kGradRows;
#pragma unroll
        for (int i = 0; i < UA; ++i) sa[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xs, xa[i], r0 * M * 2, 0));
#pragma unroll
        for (int i = 0; i < UB; ++i) sb[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(gs, gb[i], r0 * N * 2, 0));
    };
    auto load_first = [&]() __attribute__((always_inline)) {   // zeros in the place of rows before the first
        const int r0 = first + min(team, n - 1) * kGradRows;
#pragma unroll
        for (int i = 0; i < UA; ++i)
            sa[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xs, xa[i] + max(r0, -ra[i]) * M * 2, 0, 0));
#pragma unroll
        for (int i = 0; i < UB; ++i)
            sb[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(gs, gb[i] + max(r0, -rb[i]) * N * 2, 0, 0));
#pragma unroll
        for (int i = 0; i < UA; ++i)
            if (r0 + ra[i] < 0) sa[i] = u32x4{0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < UB; ++i)
            if (r0 + rb[i] < 0) sb[i] = u32x4{0, 0, 0, 0};
    };
    auto put = [&](int half) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < UA; ++i) as[half * TA + wa[i]] = sa[i];
#pragma unroll
        for (int i = 0; i < UB; ++i) bs[half * TB + wb[i]] = sb[i];
    };

    const int wave = __builtin_amdgcn_readfirstlane(tid / kBlock), lane = tid % kBlock;
    const int wm = wave % 2 * 64, wn = wave / 2 * (32 * NT);
    // This lane's place in a transposing read: 16 lanes read 4 rows x 16 columns, 8 bytes each, and
    // every lane is given four rows of a column.
    const int in16 = lane % 16, row16 = in16 / 4, half8 = lane / 32, col16 = lane / 16 % 2 * 16 + in16 % 4 * 4;
    int at_a[2], at_b[NT];   // bytes
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int col = wm + 32 * i + col16;
        at_a[i] = (8 * half8 + row16) * (CA * 16) + grad_piece<BM>(row16, col / 8) * 16 + col % 8 * 2;
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int col = wn + 32 * j + col16;
        at_b[j] = (8 * half8 + row16) * (CB * 16) + grad_piece<BN>(row16, col / 8) * 16 + col % 8 * 2;
    }
    auto fragment = [&](const u32x4_alias *base, int at, int pitch, int k) __attribute__((always_inline)) {
        const char *const from = reinterpret_cast<const char *>(base) + at + k * 16 * pitch;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)from);
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(from + 4 * pitch));
        const u32x2 l = __builtin_bit_cast(u32x2, lo), h = __builtin_bit_cast(u32x2, hi);
        return u32x4{l[0], l[1], h[0], h[1]};
    };
    f32x16 acc[2][NT] = {};
    auto multiply = [&](int half) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kGradRows / 16; ++k) {
            u32x4 a[2], b[NT];
#pragma unroll
            for (int i = 0; i < 2; ++i) a[i] = fragment(as + half * TA, at_a[i], CA * 16, k);
#pragma unroll
            for (int j = 0; j < NT; ++j) b[j] = fragment(bs + half * TB, at_b[j], CB * 16, k);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = mfma32<T>(b[j], a[i], acc[i][j]);
        }
    };

    load_first();
    put(0);
    if (mine > 1) load(1);
    lds_barrier();
    for (int t = 0; t + 1 < most; ++t) {   // tile t is in LDS, tile t + 1 in registers or on its way there
        multiply(t & 1);
        put((t + 1) & 1);
        load(min(t + 2, mine - 1));
        lds_barrier();
    }
    if (most == mine) multiply((most - 1) & 1);

    // each team hands half of its sums to the other and adds what it is handed to the half that it keeps
    lds_barrier();
    f32x4_alias *const pass = reinterpret_cast<f32x4_alias *>(memory) + tid;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const f32x16 &half = team ? acc[0][j] : acc[1][j];
            pass[((team * NT + j) * 4 + e) * kGradTeam] = f32x4{half[4 * e], half[4 * e + 1], half[4 * e + 2], half[4 * e + 3]};
        }
    lds_barrier();
    float *const out = p.out + (int64_t)split * M * N;
    const int m = m0 + wm + 32 * team + lane % 32;
    if (m >= M) return;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int col = n0 + wn + 32 * j + 8 * e + 4 * half8;
            const f32x16 &half = team ? acc[1][j] : acc[0][j];
            const f32x4 other = pass[(((1 - team) * NT + j) * 4 + e) * kGradTeam];
            if (col < N)
                *reinterpret_cast<f32x4 *>(out + (int64_t)m * N + col) =
                    f32x4{half[4 * e], half[4 * e + 1], half[4 * e + 2], half[4 * e + 3]} + other;
        }
}

// The slices' sum, in their order, in float or in 16 bits.
template <typename T>
__global__ void __launch_bounds__(256) add_slices(const float *slices, int64_t count, int splits, void *out) {
    for (int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4; i < count; i += (int64_t)gridDim.x * 1024) {
        f32x4 sum = *reinterpret_cast<const f32x4 *>(slices + i);
        for (int s = 1; s < splits; ++s) sum += *reinterpret_cast<const f32x4 *>(slices + s * count + i);
        if constexpr (sizeof(T) == 4) *reinterpret_cast<f32x4 *>(static_cast<float *>(out) + i) = sum;
        else *reinterpret_cast<u32x2 *>(static_cast<uint16_t *>(out) + i) = u32x2{pack_pair<T>(sum[0], sum[1]), pack_pair<T>(sum[2], sum[3])};
    }
}

template <typename T> hipError_t grad_of(const GradParams &p, const GradPlan &plan, hipStream_t st) {
    const void *f = plan.tile_n == 192 ? reinterpret_cast<const void *>(product_grad<T, 3>) : reinterpret_cast<const void *>(product_grad<T, 2>);
    const int64_t tiles = (int64_t)((p.inner + kGradTileM - 1) / kGradTileM) * ((p.cols + plan.tile_n - 1) / plan.tile_n);
    void *args[] = {const_cast<GradParams *>(&p)};
    return hipLaunchKernel(f, dim3((unsigned)((tiles * p.splits + 7) / 8 * 8)), dim3(kGradThreads), args, 0, st);
}

}  // namespace

hipError_t launch_product_grad(GradParams p, const GradPlan &plan, bool half, int32_t out_dtype, void *out, hipStream_t st) {
    const bool whole = p.splits == 1 && out_dtype == SRU_AMD_F32;   // the only slice is the result
    if (whole) p.out = static_cast<float *>(out);
    const hipError_t e = half ? grad_of<half_bits>(p, plan, st) : grad_of<bf16_bits>(p, plan, st);
    if (e != hipSuccess || whole) return e;
    int64_t count = (int64_t)p.inner * p.cols;
    const float *slices = p.out;
    int splits = p.splits;
    void *args[] = {&slices, &count, &splits, &out};
    const void *f = out_dtype == SRU_AMD_F32   ? reinterpret_cast<const void *>(add_slices<float>)
                    : out_dtype == SRU_AMD_F16 ? reinterpret_cast<const void *>(add_slices<half_bits>)
                                               : reinterpret_cast<const void *>(add_slices<bf16_bits>);
    const int64_t groups = (count / 4 + 255) / 256;
    return hipLaunchKernel(f, dim3((unsigned)(groups < 2048 ? groups : 2048)), dim3(256), args, 0, st);
}

}  // namespace sru_amd

// One time step of a stack of equal layers in 16-bit weights without gradients, in one launch: a token generated through all
// of its layers.
//
// What bounds it: the step kernels (layer_step.hip) took ten layers of 2048 features (projection 512, 16 rows) 20 launches that
// wait for each other, 5.4 and 7.9 us each, of which the weights' way from memory is a quarter. Here a workgroup takes
// pieces of work in the order in which they depend on each other and has a piece's weights on their way before what
// the piece reads exists: 134 -> 69 us a pass, 49 with one row (134), 174 with 64 (236); 2048 features without a projection, 8 layers, 95 -> 65;
// six layers of 512 features 64 -> 22. Recorded in a graph 106 -> 65 (8 layers); few narrow layers without projections are
// slower so and go one by one there (stack_wanted_in_graph).
// What bounds it now, per layer and 16 rows, 6.2 us: handing 64 KB of outputs and 16 KB of projected rows over, 1.5 and 1.0 us;
// from the arrival to the store 1.2 us each, of which the matrix instructions are a tenth and the partial sums' way through LDS half.
//
// Pieces. Per layer there are n_proj / 32 pieces that project 32 columns each, and Dp / 32 that make U for 32 cells (float, in
// the accumulators) and run the step on it: numbered in this order, so that a piece only reads what pieces of smaller
// numbers write. A workgroup draws its next number from a counter; the smallest unfinished number is always a running
// workgroup's current piece, so every wait ends, however few workgroups the chip has room for.
//
// Handing over. What one piece leaves for another goes through a buffer that holds a pattern no piece ever writes
// (kNotYet in every 32-bit word): stores go past the XCD's own L2 and whoever reads a word loads it the same way until
// it is there. No flags and no fences, since a word is its own flag: 1.7 us from one stage of 16 KB to the next
// with 128 workgroups (2.4 with 64 KB), 4.0 with a flag behind the data (5.2), 7 with a launch.
//
// A piece is mapped as in layer_step.hip (and gives the same sums): 8 wavefronts split the inner dimension, partial sums meet
// in LDS in wavefront order.
#include "sru_amd.h"

#include <hip/hip_runtime.h>

#include "sru_stack.h"

namespace sru_amd {
namespace {

template <typename T, int NB>
__global__ void __launch_bounds__(kStackThreads) layer_stack(const StackParams p) {
    __shared__ float parts[kStackParts];
    __shared__ StackControl control;
    if (threadIdx.x == 0) control = StackControl{draw_piece(p), kPatience};
    __syncthreads();
    int number = __builtin_amdgcn_readfirstlane(control.next);
    while (number < p.pieces) {
        int drawn = 0;
        if (threadIdx.x == 0) drawn = draw_piece(p);
        const int n_project = again(p.n_proj) / kCells, each = n_project + again(p.Dp) / kCells;
        const int l = number / each, i = number % each;
        if (i < n_project) piece<T, 2, NB, NB == 4 ? 4 : 8, true>(p, parts, control, l, i, 0, again(p.rows));
        else piece<T, 6, NB, NB == 4 ? 2 : 4, false>(p, parts, control, l, i - n_project, 0, again(p.rows));
        if (threadIdx.x == 0) control.next = drawn;
        __syncthreads();
        number = __builtin_amdgcn_readfirstlane(control.next);
    }
}

__global__ void __launch_bounds__(256) fill_not_yet(u32x4 *to, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) to[i] = u32x4{kNotYet, kNotYet, kNotYet, kNotYet};
}

template <typename T> const void *kernel_of(int rows) {
    return rows <= 16   ? reinterpret_cast<const void *>(layer_stack<T, 1>)
           : rows <= 32 ? reinterpret_cast<const void *>(layer_stack<T, 2>)
                        : reinterpret_cast<const void *>(layer_stack<T, 4>);
}

}  // namespace

hipError_t clear_exchange(StackParams &p, void *workspace, size_t bytes, hipStream_t st) {
    p.ticket = static_cast<uint32_t *>(workspace);
    p.exchange = static_cast<char *>(workspace) + kStackHeader;
    u32x4 *to = static_cast<u32x4 *>(workspace);
    int64_t n = (int64_t)(bytes / 16);
    void *args[] = {&to, &n};
    return hipLaunchKernel(reinterpret_cast<const void *>(fill_not_yet), dim3((unsigned)min((n + 255) / 256, (int64_t)2048)), dim3(256), args, 0, st);
}

// Workgroups: those of the layer at work and as many again that wait for it with their weights there already. More of them
// only ask the memory for results that are far off: with 256 (or all pieces, if fewer) / this many, us a pass:
//   2048 -> 512, 10 layers, 16 rows 71.3/69.4, 64 rows 177.3/174.5, one 48.4/48.9    1024 -> 256, 8 layers 47.4/43.1
//   1536 -> 384, 8 layers 46.1/42.8    2048, 8 layers 69.7/65.1, one row 58.7/55.1   1280, 40 rows 65.9/63.0
// Without a projection in between, a layer of few pieces is over before the weights of the next but one have arrived: as many
// again, up to 128 in all (1024, 8 layers 36.3, 34.2 with two layers' and 30.9 with three; 512, 10 layers 33.6, 33.4, 31.0).
// Below 48 there is nothing to gain (128, 16 layers 33.4 with 64, 35.7 with 12).
static int stack_workgroups(const StackParams &p) {
    const int each = p.n_proj / kCells + p.Dp / kCells;
    const int ahead = p.n_proj ? 2 * each : min(3 * each, max(2 * each, 128));
    return min(p.pieces, min(256, max(48, ahead)));
}

hipError_t launch_layer_stack(StackParams p, void *workspace, size_t bytes, bool half, hipStream_t st) {
    p.pieces = p.layers * (p.n_proj / kCells + p.Dp / kCells);
    const hipError_t e = clear_exchange(p, workspace, bytes, st);
    if (e != hipSuccess) return e;
    void *args[] = {&p};
    return hipLaunchKernel(half ? kernel_of<half_bits>(p.rows) : kernel_of<bf16_bits>(p.rows), dim3((unsigned)stack_workgroups(p)), dim3(kStackThreads), args, 0, st);
}

}  // namespace sru_amd

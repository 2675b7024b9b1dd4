// What the entry point of a whole layer hands to the kernels behind it.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sru_amd {

// One time step (layer_step.hip): rows (rows, inner) times weight (inner, cols).
struct StepParams {
    const void *x, *weight;
    const void *wc, *bias, *c0, *scale_x, *skip;
    const uint8_t *pad;
    void *h, *c_last;      // h: the product itself when it is the projection
    int64_t cols, Dp;
    int32_t rows, inner, act;
    uint32_t small16;
};

constexpr int kStepMaxRows = 64;   // four tiles of 16 rows share a weight operand
// 32 cells per workgroup, 32 inner indices per matrix instruction.
//
// The inner sizes end where the library's products are faster both for a caller that launches each call (its
// products cost 18 us of host time each, these kernels 4) and in a recorded graph. Per layer, bf16, ten
// layers, us, kernels against library products and scan, first in a graph, then launched one by one:
//                                      16 rows              32 rows              64 rows
//   1024 inner, 3072 columns         7.1/11.0  8.8/26.9   8.8/12.3  8.8/26.9  13.0/13.2 12.6/27.1
//   2048, 6144                      12.4/15.1 12.2/27.2  15.5/15.6 15.1/28.7  21.3/17.1 21.3/27.3
//   2560, 7680                      24.0/20.7 23.6/27.2  28.4/22.5 27.8/27.4  34.2/25.2 33.8/27.4
//   4096, 12288                     34.4/29.7            39.4/31.9            49.3/39.0
//   projections (against a library projection in front of the kernel):
//   2048 -> 512                     12.6/13.9 12.6/27.3  15.8/15.7 15.5/27.4  22.6/22.4 22.3/27.3
//   3072 -> 768                     18.4/16.3 18.0/27.5  23.8/20.8 23.4/27.4  31.3/30.9 30.9/30.6
//   4096 -> 1024                    29.3/27.4 28.9/27.5  35.2/30.5 34.7/30.4  46.9/43.9 46.4/43.8
// Without a limit one row of 8192 inner indices and 2048 columns took 47.5 us where library products and scan
// with converted small tensors had taken 42.6 (64 rows: 82.9 against 71.1). Between 1280 and 2048 inner
// indices 33 to 64 rows are 10-26% slower than the library in a graph and 30-50% faster launched one by one.
inline bool step_sizes_ok(int64_t rows, int64_t Dp, int64_t in_features, int64_t n_proj) {
    const int64_t product = n_proj ? n_proj : in_features, projection = n_proj ? in_features : 0;
    return rows <= kStepMaxRows && Dp % 32 == 0 && in_features % 32 == 0 && n_proj % 32 == 0 &&
           product <= (rows <= 16 ? 3072 : rows <= 32 ? 2560 : 2048) && projection <= (rows <= 16 ? 4096 : rows <= 32 ? 3072 : 2560);
}
hipError_t launch_layer_step(const StepParams &p, const StepParams *proj, bool half, int k, int skip, hipStream_t st);

// Whole sequences with the weights in registers (layer_rows.hip): x (L * B, inner) times weight
// (inner, Dp * k).
struct RowsParams {
    const void *x, *weight;
    const void *wc, *bias, *c0, *scale_x, *skip;
    const uint8_t *pad;
    void *h, *c_last;
    int64_t B, Dp;
    int32_t L, d, dirs, inner;
    int32_t groups_per_dir;   // of 64 cells
    uint32_t small16;
};

// Whether the walk is worth it, and with how many steps per matrix tile (4 or 2; 0: no walk, two calls).
//
// A walk's time goes with rounds of workgroups, not with columns: a workgroup takes 64 cells of one
// direction (a last one that is not full repeats cells) for 16 / steps batch elements, those of the same
// batch elements share one of the 8 XCDs, an XCD has 32 CUs, and a wavefront's steps follow each other.
// Per step of a round (MI355X, f16, 512 steps, 256 workgroups): inner size up to 128 160 ns with four steps
// per tile and 235 with two; up to 256 200 / 305 with three streams and 200 / 315 with four; up to 512
// 270 / 435. A further round on a CU costs as much again where the weights leave registers for one
// wavefront per SIMD (four streams over 128, three over 256), and 110-210 ns where two or three fit beside
// each other. Product and scan take time by the column: 4 ps a step plus what the product's operations
// take, 2.4 ps more where the product's last 256-wide tile is not full, and 50 ps per row of any width.
//
// The constants are fitted to 658 measured points (31 layers of 8 to 1024 cells, 49152 to 393216 columns, 256
// to 2048 steps), each with both tiles and as two calls. Deciding by columns alone was more than 5% behind
// the best of the three at 134 of them (29 times behind two calls), by up to 38%; this rule is at 4, by up
// to 11%. At 160 other random sizes: 29 by up to 39%, and 1 by 5.4%. 512 steps, two calls / two steps per
// tile / four: 133120 columns (inner 512, 256 + 256 cells) 412 / 449 / 394 us; 49248 (288, 144 + 144)
// 190 / 219 / 262; 98208 of the same 325 / 441 / 391; 163840 (256, 256 + 256, four streams) 477 / 321 / 301.
constexpr int64_t kRowsMinColumns = 49152, kRowsMinSteps = 256;   // (fewer: two calls are near or faster, or not measured)
inline int rows_steps_per_tile(int64_t B, int64_t d, int64_t dirs, int64_t inner, int k) {
    struct Cost { int first4, more4, first2, more2; };   // ns per step: one round, each further one
    const Cost c = inner <= 128 ? Cost{155, 115, 230, 155} : inner > 256 ? Cost{262, 262, 435, 435}
                   : k == 3 ? Cost{185, 145, 290, 210} : Cost{196, 196, 308, 308};
    const auto rounds = [&](int64_t per_group) {   // of the XCD that has most
        return (((B + per_group - 1) / per_group + 7) / 8 * dirs * ((d + 63) / 64) + 31) / 32;
    };
    const int64_t four = c.first4 + c.more4 * (rounds(4) - 1), two = c.first2 + c.more2 * (rounds(8) - 1);
    const int64_t columns = B * d * dirs;
    const int64_t calls = columns * (4000 + inner * k * 8 / 5 + (d * dirs * k % 256 ? 2400 : 0)) / 1000000 + B * 50 / 1000;
    return (four <= two ? four : two) > calls ? 0 : four <= two ? 4 : 2;
}
inline bool rows_sizes_ok(int64_t L, int64_t B, int64_t d, int64_t dirs, int64_t inner, int k) {
    return d % 8 == 0 && inner % 32 == 0 && inner <= (k == 3 ? 512 : 256) && L < (1 << 30) &&
           B * d * dirs >= kRowsMinColumns && L >= kRowsMinSteps &&
           B * d * dirs < (1 << 28) && B * inner < (1 << 28) &&   // (a tile's addresses are 32-bit offsets from its first time)
           rows_steps_per_tile(B, d, dirs, inner, k) != 0;
}
hipError_t launch_layer_rows(const RowsParams &p, bool half, int k, hipStream_t st);

// One time step of a stack of layers of one width in one launch (layer_stack.hip).
constexpr int kStackMaxLayers = 16;   // their pointers are kernel arguments
constexpr size_t kStackHeader = 256;  // bytes of the workspace in front of what pieces hand over
struct StackLayer {
    const void *weight, *weight_proj, *wc, *bias, *scale_x;
};
struct StackParams {
    StackLayer layer[kStackMaxLayers];
    const void *x, *c0;       // (rows, Dp); (layers, rows, Dp) or null
    const uint8_t *pad;
    void *h, *c_last;
    uint32_t *ticket;
    char *exchange;           // projected rows of every layer, outputs of every layer but the last, states between chunks
    int64_t outputs_at, states_at;
    int32_t layers, rows, Dp, n_proj, pieces, act, skip;
    uint32_t small16;
    int32_t batch, steps, chunks;   // of a sequence: rows is length * batch
    int32_t stride, delay;          // and its order of pieces (PromptOrder)
    int32_t projecting_last;
};
// Where the step kernels take each of the layers, of which there have to be two. Layer by layer / in one launch, bf16, us a pass,
// launched one by one and in a graph (8 layers unless another number is given):
//                          1 row                  16 rows                 64 rows
//   64                  82/21   27/25          82/23   29/29           81/48   51/53
//   1024                81/26   54/32          81/32   61/38          102/79  106/86
//   2048                84/56   87/62          93/64   96/70          154/127 157/134
//   2048 -> 512        108/41   94/47         109/59  106/65          181/143 184/149
//   2048 -> 512, ten   133/49  115/56         136/71  130/77          225/177 228/182
//   3072               187/142 191/147        209/167 212/172         (past the step kernels' sizes)
//   two of 64           27/15   18/18          27/15   19/19           28/16   19/21
//   two of 2048         27/20   28/27          28/23   30/29           42/37   46/44
inline bool stack_sizes_ok(int64_t layers, int64_t rows, int64_t Dp, int64_t n_proj) {
    return layers >= 2 && layers <= kStackMaxLayers && n_proj < Dp && step_sizes_ok(rows, Dp, Dp, n_proj);
}
// ... and whether it is the faster way in a graph as well, where a launch costs its host nothing. Without projections few narrow layers are over
// before the fill in front of them has paid off: a launch saves 0.6 us a layer and 1.6 more for 1000 features, less 10 ns a row, and the fill
// costs 2.5, fitted to 762 sizes in a graph (2 to 16 layers of 32 to 2048, 1 to 64 rows). The 566 on this side take 0.83 of the time, the
// worst 1.10 (32, six layers, 16 rows 22.1 / 24.3); of the 196 others 140 took longer, up to 1.19 (32, three layers, 48 rows 21.2 / 25.3). Launched one by
// one all of them gain (37.0 / 17.8), as do all with projections in a graph.
inline bool stack_wanted_in_graph(int64_t layers, int64_t rows, int64_t Dp, int64_t n_proj) {
    return n_proj > 0 || layers * (610 + 8 * Dp / 5 - 10 * rows) >= 2800;
}
// A sequence of a few batch rows through such a stack (prompt_stack.hip): time steps in a chunk, 0 where the layers one
// by one are as fast or nearly so.
//
// What it saves is the walk that follows the walk of the layer before, per layer; what it costs is products in pieces of 64 rows
// and less, and words that every layer hands over. Both ways are estimated, in ns. Layer by layer: launches, 33 ns a step, and
// products that read their weights and go at 2 PFLOP/s in the end, with the streams of the recurrence. In chunks: the way through
// the layers, which the first chunk goes alone, then what follows each other from chunk to chunk (the walk's steps; more where
// projections lie between and chunks are on their way in all layers), and the pieces of all layers on 256 compute units.
//
// Both are fitted to 10 892 points drawn at random, each measured in a graph layer by layer, in chunks of 64 rows and of 32 (three to
// sixteen layers of 32 to 2048, projections up to 3/4, one to four rows, 32 to 4096 steps): standard deviations 4.6, 7.3 and 6.1%.
// (An estimate fitted to 260 points of up to 1024 steps was up to 2.0 times slower than the layers one by one beyond them: 3550 x 3,
// 13 layers of 2048 -> 512, 2959 -> 6021 us.) Where the better of the chunks is expected to take 0.93 of the time it takes 0.66 of it, over
// 8 270 points; 0.9% of these take longer, 0.4% by more than 5%, the worst 1.27 (644 x 3, 13 layers of 1792 -> 448, 730 us layer by layer).
// Launched one by one, a layer costs its host 12.4 us, 16 with a projection, of which 12 and 14 are counted on, and the launches here
// take 7 us less than in a graph: three layers of 64, 32 steps, 47 us and 26, where a graph takes 34 and 33. Of 2 930 points of up to 600 steps
// that are taken 4 are slower launched so, the worst 1.14. (3 803 further points that are taken, in a graph: 0.67, 3% slower, the worst 1.13.)
// Layer by layer / chunks of 64 rows / 32, bf16, us a pass in a graph:
//   one row   512 x 2048 -> 512, 10 layers 424/286/320    1024 of the same 640/496/628   128 of the same 229/163/144
//             370 x 256, 10 layers 207/119/93     491 x 1024, 6 layers 215/139/133  230 x 512 -> 128, 4 layers 79/67/58
//             936 x 2048 -> 512, 10 layers 606/457/589    54 x 2048 -> 512, 8 layers 171/131/112
//   two rows  512 x 512, 4 layers 119/77/82       175 x 1280 -> 320, 10 layers 247/237/171
//   three     276 x 384, 6 layers 122/86/89       104 x 2048 -> 512, 8 layers 211/171/192
//   four      143 x 384 -> 96, 10 layers 171/139/139      346 x 2048 -> 512, 10 layers 510/605/814
constexpr int kStackRows = 64;        // rows of a chunk at the most
struct ChunkCost {
    int launch, layer, layer_projects, layer_step, chunk, chunk_waits, step, walk, walk_more, project;   // walk_more: past what LDS holds at once
};
inline int prompt_steps(int64_t layers, int64_t length, int64_t batch, int64_t Dp, int64_t n_proj) {
    const int64_t inner = n_proj ? n_proj : Dp, weights = n_proj ? 4 * Dp * n_proj : 3 * Dp * Dp;
    if (layers < 3 || layers > kStackMaxLayers || length < 32 || length > 4096 || batch > 4 || Dp % 32 != 0 || n_proj % 32 != 0 || n_proj >= Dp || Dp > 2048 ||
        inner > (length >= 256 ? 1024 : 512))
        return 0;
    const int64_t one_by_one = 8600 + layers * (6300 + (n_proj ? 3000 : 0) + 33 * length + weights / 300 + length * batch * (weights + 6300 * Dp) / 1000000);
    const auto in_chunks = [&](int64_t rows, int64_t stride, const ChunkCost &c) {
        const int64_t steps = rows / batch, chunks = (length + steps - 1) / steps, walks = (Dp + 63) / 64, projections = n_proj / 32 * (rows / 32);
        const int64_t waiting = n_proj && chunks > layers * stride ? chunks - layers * stride : 0;
        return c.launch + layers * (c.layer + (n_proj ? c.layer_projects : 0) + c.layer_step * steps) + chunks * c.chunk + waiting * c.chunk_waits + length * c.step +
               chunks * layers * (walks * (c.walk + (inner > 512 ? c.walk_more : 0)) + projections * c.project);
    };
    const int64_t wide = in_chunks(kStackRows, 3, ChunkCost{12000, 6570, 1800, 31, 745, 1120, 34, 31, 29, 26});
    const int64_t narrow = in_chunks(kStackRows / 2, 4, ChunkCost{14000, 4450, 1680, 37, 650, 390, 31, 21, 27, 32});
    const int64_t best = wide < narrow ? wide : narrow, launched = 10000 + layers * (n_proj ? 14000 : 12000);
    return best * 100 > (one_by_one < launched ? launched : one_by_one) * 93 ? 0 : (int)((wide < narrow ? kStackRows : kStackRows / 2) / batch);
}
// A workspace holds what every layer hands over, over the whole sequence, and is filled and written once and read once each pass: where it
// no longer fits beside the weights in the last-level cache the pieces wait for memory (10 layers of 2048 -> 512 reach this
// at 4270 rows). Layer by layer two layers' worth are held.
constexpr size_t kStackMaxBytes = (size_t)192 << 20;
struct StackPlan {
    int steps, chunks;
    int64_t outputs_at, states_at;
    size_t bytes;
};
inline StackPlan stack_plan(int64_t layers, int64_t length, int64_t batch, int64_t Dp, int64_t n_proj) {
    StackPlan plan{};
    plan.steps = length == 1 ? (int)stack_sizes_ok(layers, batch, Dp, n_proj) : prompt_steps(layers, length, batch, Dp, n_proj);
    if (plan.steps == 0) return plan;
    const int64_t rows = length * batch;
    plan.chunks = (int)((length + plan.steps - 1) / plan.steps);
    plan.outputs_at = layers * rows * n_proj * 2;
    plan.states_at = plan.outputs_at + (layers - 1) * rows * Dp * 2;
    plan.bytes = kStackHeader + (size_t)(plan.states_at + layers * (plan.chunks - 1) * batch * Dp * 4);
    return plan.bytes > kStackMaxBytes ? StackPlan{} : plan;
}
// The order in which a prompt's pieces are numbered. A slot has the projecting pieces of one chunk of every `stride`-th
// layer and then the walking ones `delay` chunks behind; of a slot's layers only the lowest can be at the last chunk, which
// has fewer projecting pieces where it has fewer rows. There is no piece without rows: whoever runs one passes a barrier in it.
struct PromptOrder {
    int layers, chunks, stride, delay;
    int projecting, projecting_last, walking;   // pieces of a chunk, and of the last one
};
struct PromptPiece {
    int layer, chunk, index;   // index: among the chunk's pieces of its kind
    bool project;
};
inline PromptOrder prompt_order(const StackParams &p) {
    const int halves = p.steps * p.batch <= 32 ? 1 : 2, columns = p.n_proj / 32;   // (projecting pieces have 32 rows, chunks two halves)
    const int last = p.rows - (p.chunks - 1) * p.steps * p.batch;
    const int stride = halves == 1 ? 4 : 3;
    return {p.layers, p.chunks, stride, p.n_proj ? stride - 2 : 0, columns * halves, columns * ((last + 31) / 32), (p.Dp + 63) / 64};
}
inline int prompt_pieces(const PromptOrder &o) {
    return o.layers * ((o.chunks - 1) * o.projecting + o.projecting_last + o.chunks * o.walking);
}
// Piece `number`, which has to be one; slot and before (the number of pieces in slots in front of it) start from zero and are those of
// the last piece asked for, of a smaller number.
__host__ __device__ inline PromptPiece prompt_piece(const PromptOrder &o, int number, int &slot, int &before) {
    const auto less = [](int a, int b) { return a < b ? a : b; };
    const auto more = [](int a, int b) { return a < b ? b : a; };
    for (;;) {   // (ends: `number` is that of a piece of some slot)
        const int first = more(0, (slot - o.chunks + o.stride) / o.stride), first_walk = more(0, (slot - o.delay - o.chunks + o.stride) / o.stride);
        const int layers = more(0, less(slot / o.stride, o.layers - 1) - first + 1);
        const int walks = slot < o.delay ? 0 : more(0, less((slot - o.delay) / o.stride, o.layers - 1) - first_walk + 1);
        const int absent = layers > 0 && slot - first * o.stride == o.chunks - 1 ? o.projecting - o.projecting_last : 0;
        const int projects = layers * o.projecting - absent;
        int i = number - before;
        if (i < projects) {
            if (i >= o.projecting - absent) i += absent;
            return {first + i / o.projecting, slot - (first + i / o.projecting) * o.stride, i % o.projecting, true};
        }
        i -= projects;
        if (i < walks * o.walking) {
            const int layer = first_walk + i / o.walking;
            return {layer, slot - o.delay - layer * o.stride, i % o.walking, false};
        }
        before += projects + walks * o.walking;
        ++slot;
    }
}
hipError_t clear_exchange(StackParams &p, void *workspace, size_t bytes, hipStream_t st);   // and sets where it is
hipError_t launch_prompt_stack(StackParams p, void *workspace, size_t bytes, bool half, hipStream_t st);
hipError_t launch_layer_stack(StackParams p, void *workspace, size_t bytes, bool half, hipStream_t st);

// A product by itself (product.hip): x (rows, inner) times weight (inner, cols), all in one type.
struct ProductParams {
    const void *x, *weight;
    void *out;
    int32_t rows, inner, cols;
};

// The tile of a product's workgroups, 32 rows x 32 columns at the least, and whether they split the inner dimension
// in two; none where a size is not a whole number of 16-byte pieces or the library's product is the faster one by far.
//
// Larger tiles read less, smaller ones leave a workgroup for more compute units: a larger one is taken from about
// three workgroups to four compute units on (float, whose tiles take four times as long in the matrix cores, from
// three workgroups to a unit), unless that is just one round of them and a little of another, of many inner indices
// each: tiles of 32 x 64 then are two rounds (bf16 200 x 1024 -> 4416, 276 workgroups 12.7 us, 32 x 64 tiles 10.1, library 11.5;
// 136 x 1792 -> 5632 19.4, 16.8, 17.3) or more, and level. Two halves of the inner dimension where it is long and compute units are left over.
// Measured (us in a graph, library / 32 x 32 / 32 x 64 / 64 x 64, the rule's choice marked *, with "2" where split):
//   bf16   33 x 256 -> 768      4.5/3.1*/3.6/3.9      128 x 256 -> 3072    6.7/4.0/3.8*/4.4    512 x 512 -> 6144   12.9/17.1/13.4/11.3*
//          128 x 1024 -> 256    10.5/4.8*2/6.3/7.4    512 x 2048 -> 512   10.8/8.8*2/10.3/12.6 128 x 2048 -> 6144  18.8/17.7/16.1/13.1*2
//   f32    640 x 128 -> 384     4.3/3.4*/4.3/5.6      2048 x 256 -> 768   22.3/12.3/12.2*/14.0 1024 x 256 -> 3072  24.7/21.0/19.6/18.9*
// Past 1.75e9 multiply-adds the library is faster (bf16 512 x 2048 -> 6144 26.4/30.5, 1024 x 512 -> 6144
// 16.3/18.8, 2048 x 1024 -> 3072 21.9/30.8). In float it is faster too where the inner dimension is long (128 x 2048 -> 512
// 10.0/14.3, 64 x 1536 -> 4608 17.2/18.8) or longer than the result is wide (512 x 1024 -> 256 8.9/9.3); below 64 inner
// indices or columns it is not measured.
struct ProductTile { int m, n, split; };   // in units of 32; m 0: none
inline ProductTile product_tile(int size, int64_t rows, int64_t inner, int64_t cols) {
    const bool f32 = size == 4;
    if (rows < 1 || inner < 1 || cols < 1 || inner % (f32 ? 4 : 8) != 0 || cols % 4 != 0 || rows > (1 << 20) || inner > (1 << 14) ||
        cols > (1 << 16) || (f32 && (inner < 64 || cols < 64)) || rows * inner * cols > (int64_t)1750000000 || (f32 && inner > 512 && (inner > 1024 || cols < 2 * inner)))
        return {0, 0, 0};
    const auto tiles = [&](int m, int n) { return (rows + 32 * m - 1) / (32 * m) * ((cols + 32 * n - 1) / (32 * n)); };
    ProductTile t = tiles(2, 2) >= (f32 ? 768 : 192) ? ProductTile{2, 2, 1} : tiles(1, 2) >= (f32 ? 384 : 192) ? ProductTile{1, 2, 1} : ProductTile{1, 1, 1};
    if (!f32 && inner >= 1024 && t.m == 2 && tiles(2, 2) > 256 && tiles(2, 2) <= 320) t.m = 1;
    if (inner >= (f32 ? 512 : 1024) && tiles(t.m, t.n) <= 256) t.split = 2;
    return t;
}
// Whether a layer's product is made by the kernel: up to where, over sizes drawn at random, its time in a graph is still the
// shorter one on average. In 16 bits that is a matter of the result's size, the sooner the more inner indices there are:
// 375 sizes on this side 0.77 of the library's time, the worst 1.30 (4502 x 320 -> 768 9.6/12.5); 196 beyond level, the worst
// 1.66 (777 x 640 -> 1920 9.6/10.5, 3007 x 128 -> 3584 12.1/17.1). In float it is one of work at more than 384 inner indices:
// 216 sizes 0.78, the worst 1.26 (2855 x 512 -> 384 15.9/20.0), beyond 1.03 and 1.35. Launched one by one a library product
// costs its caller 18 us, and this one 4, which is why the line lies no lower.
inline bool product_wanted(int size, int64_t rows, int64_t inner, int64_t cols) {
    if (product_tile(size, rows, inner, cols).m == 0) return false;
    if (size == 4) return inner <= 384 || rows * inner * cols <= 600000000;
    return rows * cols <= (inner <= 512 ? 3500000 : 1000000);
}
hipError_t launch_product(const ProductParams &p, int32_t dtype, const ProductTile &tile, hipStream_t st);

// The gradient of a product's weight (product_grad.hip): x (rows, inner) transposed times g (rows, cols), both in 16
// bits, as float slices (splits, inner, cols) of parts of the rows.
struct GradParams {
    const void *x, *g;
    float *out;
    int32_t rows, inner, cols, splits;
};

// The tile of the workgroups (128 columns of x by tile_n of g) and the number of parts of the rows; 0: the library's
// product is not slower, or a size is not a whole number of 16-byte pieces.
//
// At most one round of workgroups, one to each of 256 compute units: a pair of tiles of 64 rows takes 1.12 us with 128
// columns and 1.52 with 192, the slices are written and read at 2.5 TB/s, and the sum of both is least. Measured (us,
// library product with conversion / 128 columns / 192, with the best number of parts each, the rule's choice marked *):
//   8192 rows   512 x 6144   92/77/65*      2048 x 512   56/30*/33    1024 x 3072  83/73/63*    256 x 1024  54/20*/23
//   4096 rows   512 x 1536   30/22*/24      256 x 3008   34/20*/22    1024 x 3072  49/43/40*
//   16384 rows  512 x 3072   125/72/63*     10195 rows, 1152 x 976  89/40*/43
// More rows and smaller results are the library's worst (38185 rows, 568 x 688 240 -> 51).
// 67 sizes drawn at random that are split take 0.40 of the library's time, the worst 0.82. Rows that are not split take
// one launch where the gradient is float. With 192 columns they take 0.75 of its time over 28 sizes (9682 rows, 1024 x
// 4384 188 -> 112; 3782 rows, 1552 x 2480 58 -> 52), but from 25000 rows on, where the library's larger tiles settle in,
// five sizes lie between 0.78 and 1.17 (32951 rows, 1016 x 4544 340 -> 396) and are left to it, as is what 128 columns
// would be better for (0.73 to 0.89). Beyond one round it is faster (16384 rows, 2048 x 6144 362 / 453).
struct GradPlan { int tile_n, splits; };
// A call costs its host some 25 us more than torch's: taken from 8192 rows on, where the library loses more than that
// (8192 rows, 256 x 256 50/17, 128 x 512 70/17; 16384 rows, 256 x 768 95/24), below where the products keep the GPU
// busier than the host (from 3000 rows and 3e9 multiply-adds; 4096 rows, 256 x 1024 30/17 is left alone). More than 16
// parts were no faster anywhere.
constexpr int64_t kGradMinRows = 3000, kGradManyRows = 8192, kGradMinWork = 3000000000, kGradMinResult = 128 * 384, kGradWholeRows = 24576;
inline GradPlan product_grad_plan(int64_t rows, int64_t inner, int64_t cols) {
    if (rows < kGradMinRows || rows > (1 << 24) || inner > (1 << 16) || cols > (1 << 16) || inner < 128 || cols < 128 || inner % 8 != 0 || cols % 8 != 0 || inner * cols < kGradMinResult ||
        (rows < kGradManyRows && rows * inner * cols < kGradMinWork) || rows * inner >= (1 << 30) || rows * cols >= (1 << 30))   // (31-bit byte offsets)
        return {0, 0};
    GradPlan best{0, 0};
    int64_t least = 0;
    for (const int tile_n : {128, 192}) {
        const int64_t tiles = (inner + 127) / 128 * ((cols + tile_n - 1) / tile_n);
        for (int64_t splits = 1; splits <= 16 && tiles * splits <= 256 && splits * 256 <= rows; ++splits) {
            const int64_t pairs = ((rows + 63) / 64 + 2 * splits - 1) / (2 * splits);
            const int64_t cost = pairs * (tile_n == 128 ? 1120 : 1520) + splits * inner * cols * 8 / 2500;   // ns
            if (best.splits == 0 || cost < least) best = GradPlan{tile_n, (int)splits}, least = cost;
        }
    }
    return best.splits == 1 && (best.tile_n == 128 || rows > kGradWholeRows) ? GradPlan{0, 0} : best;
}
// p.out: room for the slices; out: the result in out_dtype (float or the 16 bits of x and g)
hipError_t launch_product_grad(GradParams p, const GradPlan &plan, bool half, int32_t out_dtype, void *out, hipStream_t st);

}  // namespace sru_amd

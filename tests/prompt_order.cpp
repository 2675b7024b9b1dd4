// Walks the pieces of prompts as prompt_stack.hip numbers them (sru_layer.h), for test_prompt_order_host.py: every piece of every
// chunk once, none without rows, and none before what it reads.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "sru_layer.h"

using namespace sru_amd;

static void fail(const char *what, const StackParams &p, int number) {
    std::printf("%s: %d layers of %d, projection %d, %d rows in chunks of %d x %d, piece %d\n", what, p.layers, p.Dp, p.n_proj, p.rows, p.steps, p.batch, number);
    std::exit(1);
}

static void check(const StackParams &p) {
    const PromptOrder o = prompt_order(p);
    const int total = prompt_pieces(o), columns = p.n_proj / 32, rows = p.steps * p.batch, halves = rows <= 32 ? 1 : 2;
    std::vector<int> projected(p.layers * p.chunks), walked(p.layers * p.chunks);   // pieces of a layer's chunk so far
    std::vector<char> seen((size_t)p.layers * p.chunks * (columns * 2 + o.walking));
    const auto complete = [&](int l, int c) { return walked[l * p.chunks + c] == o.walking; };
    int slot = 0, before = 0;
    for (int number = 0; number < total; ++number) {
        const PromptPiece at = prompt_piece(o, number, slot, before);
        int fresh_slot = 0, fresh_before = 0;   // (of a workgroup that draws its first piece)
        const PromptPiece same = prompt_piece(o, number, fresh_slot, fresh_before);
        if (same.layer != at.layer || same.chunk != at.chunk || same.index != at.index || same.project != at.project) fail("depends on the piece before", p, number);
        if (at.layer < 0 || at.layer >= p.layers || at.chunk < 0 || at.chunk >= p.chunks || at.index < 0) fail("outside", p, number);
        const int of = at.layer * p.chunks + at.chunk, R = std::min(rows, p.rows - at.chunk * rows), here = std::min(halves, (R + 31) / 32);
        int place;
        if (at.project) {
            if (at.index >= columns * here || at.index % here * 32 >= R) fail("no rows", p, number);
            if (at.layer > 0 && !complete(at.layer - 1, at.chunk)) fail("projects before its input", p, number);
            place = at.index / here * 2 + at.index % here;
            ++projected[of];
        } else {
            if (at.index >= o.walking) fail("outside", p, number);
            if (columns ? projected[of] != columns * here : at.layer > 0 && !complete(at.layer - 1, at.chunk)) fail("walks before its input", p, number);
            if (at.chunk > 0 && !complete(at.layer, at.chunk - 1)) fail("walks before its state", p, number);
            place = columns * 2 + at.index;
            ++walked[of];
        }
        if (seen[(size_t)of * (columns * 2 + o.walking) + place]++) fail("twice", p, number);
    }
    for (int l = 0; l < p.layers; ++l)
        for (int c = 0; c < p.chunks; ++c)
            if (!complete(l, c)) fail("not all pieces", p, total);
}

int main() {
    int plans = 0, short_last = 0;
    for (const int layers : {3, 4, 7, 10, 16})
        for (const int Dp : {32, 96, 256, 480, 1024, 2048})
            for (const int n_proj : {0, 32, 64, 160, 512})
                for (const int batch : {1, 2, 3, 4})
                    for (const int length : {32, 33, 63, 64, 65, 95, 96, 97, 100, 127, 128, 129, 170, 257, 289, 513, 545, 700, 1024, 1025}) {
                        const StackPlan plan = stack_plan(layers, length, batch, Dp, n_proj);
                        if (plan.steps == 0) continue;
                        StackParams p{};
                        p.layers = layers, p.Dp = Dp, p.n_proj = n_proj, p.rows = length * batch, p.batch = batch, p.steps = plan.steps, p.chunks = plan.chunks;
                        check(p);
                        ++plans;
                        const int rows = plan.steps * batch;
                        short_last += n_proj > 0 && rows > 32 && p.rows - (plan.chunks - 1) * rows <= 32;
                    }
    std::printf("%d plans, %d with a last chunk of one half\n", plans, short_last);
    return plans < 500 || short_last < 20;
}

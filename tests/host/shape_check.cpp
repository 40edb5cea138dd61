// CPU check of the launch shape that an FP32 batch runs when none is recorded
// (default_shape in rvs_context.hpp): what a shape needs, over a grid of
// robots, scenes and batches, and the shapes measured fastest on MI355X at
// points on both sides of the rule's lines.
#include <cstdio>

#include "../../rpmplv2_amd/csrc/rvs_context.hpp"

using namespace rvs;

int main() {
    int bad = 0;
    auto need = [&](bool ok, const char* what, int links, int objects, long n, bool lists, const FastTuning& t) {
        if (ok) return;
        if (++bad <= 20)
            printf("%s: links %d objects %d n %ld lists %d -> variant %d block %d bits %d\n", what, links, objects, n,
                   (int)lists, t.variant, t.block, t.coh_bits);
    };
    for (int links = 1; links <= 64; ++links)
        for (int objects = 0; objects <= 1024; objects += objects < 40 ? 1 : 23)
            for (long n = 1; n <= (1L << 31); n = n < 64 ? n + 1 : n * 3 / 2)
                for (bool lists : {false, true}) {
                    const FastTuning t = default_shape(links, links, objects, n, lists);
                    need(t.variant == 0 || t.variant == 1 || t.variant == 3 || t.variant == 4, "variant", links,
                         objects, n, lists, t);
                    need(t.variant != 4 || (lists && fast_links_bytes(n) <= (size_t(2) << 30) + 4096),
                         "lists not to be had", links, objects, n, lists, t);
                    need(t.variant == 0 || (long)links * objects >= 1024, "long-walk shape", links, objects, n, lists, t);
                    need(t.variant >= 3 ? t.block == 512 : (t.block == 64 || t.block == 256), "block", links, objects, n,
                         lists, t);
                    need(t.blocks_per_cu == 0 && (t.coh_bits == 0 || t.coh_bits == 5), "bits", links, objects, n, lists,
                         t);
                }
    const struct {
        int links, objects;
        long n;
        bool lists;
        int variant;
    } point[] = {
        // the call cannot have lists: queues for long chains among many obstacles
        {22, 200, 1000000, false, 3}, {22, 512, 400000, false, 3}, {14, 200, 1000000, false, 3},
        {40, 200, 400000, false, 3}, {22, 200, 30000, false, 3}, {22, 128, 30000, false, 3},
        // ... and lane refill for short ones, and among fewer obstacles
        {6, 200, 400000, false, 1}, {6, 600, 1000000, false, 1}, {10, 160, 1000000, false, 1},
        {22, 128, 1000000, false, 1}, {14, 130, 1000000, false, 1},
        // link-major launches
        {22, 512, 1000, true, 4}, {22, 512, 2097152, true, 4}, {22, 200, 1000000, true, 4}, {14, 512, 30000, true, 4},
        {6, 1000, 1000000, true, 4}, {6, 200, 1000, true, 4}, {10, 400, 1000000, true, 4}, {14, 256, 1000, true, 4},
        {40, 400, 400000, true, 4}, {22, 512, 1, true, 4},
        // ... not for short chains or few obstacles
        {10, 130, 1000000, true, 1}, {10, 300, 30000, false, 1}, {10, 700, 30000, false, 3}, {6, 200, 1000000, true, 1}, {22, 200, 30000, true, 3},
        {40, 256, 30000, true, 3}, {22, 96, 400000, true, 1}, {22, 128, 1000000, true, 1}, {22, 96, 30000, true, 3}, {14, 160, 1000000, true, 3},
        // a handful of configurations
        {22, 256, 1, true, 1}, {22, 256, 10, true, 1}, {10, 130, 10, true, 1}, {40, 150, 10, true, 1},
        {22, 512, 1, false, 1}, {6, 1000, 10, false, 1},
    };
    for (const auto& p : point) {
        const FastTuning t = default_shape(p.links, p.links, p.objects, p.n, p.lists);
        need(t.variant == p.variant, "measured faster", p.links, p.objects, p.n, p.lists, t);
    }
    const struct {
        int dofs, links, objects;
        long n;
        bool sorted;
    } order[] = {
        {6, 6, 17, 1000003, true}, {6, 6, 17, 260000, false}, {6, 6, 17, 4000, false}, {10, 10, 60, 200000, false},
        {6, 6, 120, 40000, true}, {6, 6, 160, 200000, true}, {14, 14, 70, 200000, true}, {14, 14, 40, 200000, false},
        {22, 22, 1, 1000000, false}, {6, 6, 5, 4000000, false},
        {2, 2, 40, 65536, true}, {2, 2, 15, 1000000, true}, {2, 2, 15, 130000, false}, {2, 2, 4, 1000003, false},
    };
    for (const auto& p : order) {
        const FastTuning t = default_shape(p.dofs, p.links, p.objects, p.n, true);
        need((t.coh_bits > 0) == p.sorted, "measured faster", p.links, p.objects, p.n, true, t);
    }
    printf("shape_check: %d wrong\n", bad);
    return bad ? 1 : 0;
}

// Host check of which kernel a layer matrix's step takes (gpu::mm_route): no work-group is given a token tile that the
// step does not have, and a K-split step takes two token tiles per work-group only where the busiest CU's work-groups
// then take less time (measured cost of a two-tile work-group against a one-tile one: Q6_K 1.45, others 1.7-1.8). And
// which attention a step takes, against measured times.
#include "jfh_kernels.hpp"

#include <cstdio>
#include <cstdlib>

using jfh::gpu::mm_route;
using jfh::gpu::MmKernel;
using jfh::gpu::MmRoute;

namespace {

int failures = 0;

void expect(bool ok, const char* what, uint32_t type, int rows, int cols, int n) {
    if (ok) return;
    if (++failures < 20) std::printf("FAIL: %s: type %u, %d x %d, %d rows\n", what, type, rows, cols, n);
}

}  // namespace

int main() {
    for (uint32_t type : {7u, 9u, 11u, 13u}) {
        const double cost = type == 13 ? 1.45 : 1.75;
        for (int rows = 256; rows <= 60000; rows += rows < 8192 ? 256 : 1792) {
            for (int cols : {256, 512, 1536, 2048, 2304, 3584, 5120, 8960, 18944, 27648}) {
                for (int n = 9; n <= 2048; n += n < 300 ? 1 : 61) {
                    const MmRoute r = mm_route(type, rows, cols, n);
                    const int n_tt = (n + 15) / 16, n_rg = (rows + 15) / 16;
                    // as many tiles as the step has, or four for three
                    expect(r.tiles >= 1 && (r.tiles <= n_tt || (r.tiles == 4 && n_tt == 3)), "a token tile past the step",
                           type, rows, cols, n);
                    if (r.kernel != MmKernel::kFold) continue;
                    auto per_cu = [&](int tiles) { return ((n_rg + 1) / 2 * ((n_tt + tiles - 1) / tiles) + 255) / 256; };
                    if (r.groups == 2 && r.tiles == 2) {
                        expect(cost * per_cu(2) < 1.05 * per_cu(1), "two token tiles per work-group take longer", type, rows, cols, n);
                    }
                    if (r.groups == 2 && r.tiles == 1 && n_tt > 1) {
                        expect(1.05 * cost * per_cu(2) >= per_cu(1), "one token tile per work-group takes longer", type, rows, cols, n);
                    }
                }
            }
        }
    }
    // Q8_0 on grids too small for two token tiles: the faster of the two forms, as measured (us)
    struct {
        int rows, cols, n;
        double one_tile, split;
    } const q8[] = {{5120, 27648, 96, 164, 141}, {5120, 27648, 128, 188, 173}, {5120, 13824, 96, 81.0, 73.3},
                    {5120, 13824, 113, 94.4, 86.4}, {4096, 12288, 128, 78.2, 67.0}, {4096, 12288, 64, 71.1, 38.5},
                    {3584, 18944, 100, 107.5, 92.5}, {1536, 8960, 256, 46.7, 37.6}, {1536, 8960, 333, 47, 55},
                    {4608, 3584, 100, 20.4, 27.9}, {4608, 3584, 160, 25.5, 33.1}, {3584, 3584, 144, 20.3, 28.1},
                    {4096, 4096, 128, 22.9, 25.8}, {10240, 2560, 48, 18.7, 25.2}};
    for (const auto& m : q8) {
        const MmRoute r = mm_route(7, m.rows, m.cols, m.n);
        expect((r.kernel == MmKernel::kGemm && r.tiles == 1) == (m.one_tile < m.split), "the slower Q8_0 form", 7, m.rows, m.cols, m.n);
    }
    // attention of one sequence's step at a position: with key splits and without, as measured (us)
    struct {
        int heads, kv, dim, pos, rows;
        double split, whole;
    } const attn[] = {{40, 8, 128, 64, 217, 33.7, 23.7},   {40, 8, 128, 1024, 230, 71.9, 57.5},
                      {40, 8, 128, 8192, 204, 288, 303},   {40, 8, 128, 24576, 204, 716, 872},
                      {40, 8, 128, 24576, 230, 800, 880},  {40, 8, 128, 24576, 256, 884, 838},
                      {32, 32, 128, 1024, 200, 57.0, 55.9}, {32, 32, 128, 2048, 200, 81.5, 90.8},
                      {32, 32, 128, 24576, 200, 595, 869}, {64, 8, 128, 4096, 192, 233, 155},
                      {64, 8, 128, 24576, 136, 759, 832},  {64, 8, 64, 512, 128, 29.2, 25.4},
                      {64, 8, 64, 2048, 128, 50.7, 58.0},  {64, 8, 64, 8192, 160, 164, 189},
                      {64, 8, 64, 24576, 192, 498, 536},   {32, 32, 64, 4096, 200, 69.2, 109}};
    for (const auto& m : attn) {
        const bool whole = jfh::gpu::attention_prefill_supported(m.rows, 1, m.heads, m.kv, m.dim, m.pos + m.rows);
        if (whole != (m.whole < m.split)) {
            ++failures;
            std::printf("FAIL: the slower attention: %d / %d heads x %d, %d rows at %d\n", m.heads, m.kv, m.dim, m.rows, m.pos);
        }
    }
    if (failures == 0) std::printf("route tests passed\n");
    return failures == 0 ? 0 : 1;
}

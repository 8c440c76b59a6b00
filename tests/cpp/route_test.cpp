// Host check of which kernel a layer matrix's step takes (gpu::mm_route): no work-group is given a token tile that the
// step does not have, and a K-split step takes two token tiles per work-group only where the busiest CU's work-groups
// then take less time (measured cost of a two-tile work-group against a one-tile one: Q6_K 1.45, others 1.7-1.8).
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
    if (failures == 0) std::printf("route tests passed\n");
    return failures == 0 ? 0 : 1;
}

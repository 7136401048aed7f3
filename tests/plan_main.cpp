// Prints what the rules of lbm_plan.h choose, one line a request read.
#include "lbm_plan.h"

#include <cstdio>
#include <cstring>
#include <vector>

struct Size { int nx, ny; };

int main() {
    char what[16];
    while (std::scanf("%15s", what) == 1) {
        if (!std::strcmp(what, "batch")) {
            int n;
            long every;
            if (std::scanf("%d %ld", &n, &every) != 2) return 1;
            std::vector<Size> s((size_t)n);
            long tiles = 0;
            for (Size& k : s) {
                if (std::scanf("%d %d", &k.nx, &k.ny) != 2) return 1;
                tiles += ((long)k.nx * k.ny + 1023) / 1024;
            }
            const lbm::BatchPlan p = lbm::batch_plan(s.data(), n, tiles, 248, every);
            std::printf("%d %ld %d\n", p.halo, p.squares, p.grid);
        } else {
            return 1;
        }
    }
    return 0;
}

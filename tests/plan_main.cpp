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
        } else if (!std::strcmp(what, "flow2")) {
            int nx, ny, f64, mrt;
            size_t nf;
            if (std::scanf("%d %d %zu %d %d", &nx, &ny, &nf, &f64, &mrt) != 5) return 1;
            const lbm::StepPlan p = lbm::flow2_plan(nx, ny, nf, f64 != 0, mrt != 0);
            std::printf("%d %d\n", p.most, p.least);
        } else if (!std::strcmp(what, "cg2")) {
            int nx, ny, ho, enh, f64;
            if (std::scanf("%d %d %d %d %d", &nx, &ny, &ho, &enh, &f64) != 5) return 1;
            const lbm::StepPlan p = lbm::cg2_plan(nx, ny, ho != 0, enh != 0, f64 != 0);
            std::printf("%d %d\n", p.most, p.least);
        } else {
            return 1;
        }
    }
    return 0;
}

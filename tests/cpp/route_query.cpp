// Prints the kernel that a call takes (infer_amd/csrc/iq_plan.h), for the CPU
// tests of the shapes in the GPU tests.  One query a line on stdin:
//   gemm T N K kind fp32|bf16 cus part_floats
//       -> "splits" (gemm_kernel splits fp32 x itself), "narrow", or
//          "wide bm=.. full=.. splits=.. live=.." (live: 16-row blocks in use
//          of the two waves' of the last row tile, "4,1")
//   rows M tiles K kind cus part_floats
//       -> "gemvw ng=.. S=.." or "other" (and why: preferred, plan, room)
// (whole 128-column groups, aligned operands)
#include <cstdio>
#include <cstring>

#include "../../infer_amd/csrc/iq_plan.h"

int main() {
    char line[256];
    while (std::fgets(line, sizeof line, stdin)) {
        long long a, b, c, part;
        int kind, cus;
        char x[8];
        if (std::sscanf(line, "gemm %lld %lld %lld %d %7s %d %lld", &a, &b, &c, &kind, x, &cus, &part) == 7) {
            const bool lo = std::strcmp(x, "fp32") == 0;
            if (lo && iq::gemm_splits_x(a, b, c)) {
                std::puts("splits");
                continue;
            }
            const iq::GemmwPlan p = iq::gemmw_choose(a, b, c, kind, lo, cus, part);
            if (p.us > 1e29) {
                std::puts("narrow");
                continue;
            }
            int live[2];
            for (int w = 0; w < 2; w++) {
                const int mb = p.bm / 32, rows = int(a - (long long)(p.tiles_m - 1) * p.bm) - w * 16 * mb;
                live[w] = std::min(mb, (std::max(rows, 0) + 15) / 16);
            }
            std::printf("wide bm=%d full=%d splits=%d live=%d,%d\n", p.bm, p.full, p.splits, live[0], live[1]);
        } else if (std::sscanf(line, "rows %lld %lld %lld %d %d %lld", &a, &b, &c, &kind, &cus, &part) == 6) {
            const iq::GwPlan p = iq::gemvw_plan(c / 128, int(a), int(b), cus);
            if (!iq::gemvw_preferred(int(a), int(b), c, kind, cus)) std::puts("other preferred");
            else if (!p.ok) std::puts("other plan");
            else if (p.S > 1 && p.S * a * b * 16 > part) std::puts("other room");
            else std::printf("gemvw ng=%d S=%d\n", p.ng, p.S);
        } else {
            std::printf("bad query: %s", line);
            return 1;
        }
    }
    return 0;
}

// CPU checks of the wide-tile GEMM's plans (infer_amd/csrc/iq_plan.h): every
// plan covers each tile's groups once, leaves no workgroup without a group,
// and keeps its range sums inside the workspace it is given.
#include <cstdio>

#include "../../infer_amd/csrc/iq_plan.h"

static int failures = 0;

#define CHECK(c)                                                                                              \
    do {                                                                                                      \
        if (!(c)) {                                                                                           \
            std::printf("FAIL %s: T=%d N=%lld G=%d bm=%d lo=%d cus=%d part=%lld least=%d\n", #c, T, (long long)N, G, \
                        bm, lo, cus, (long long)part, least);                                                 \
            ++failures;                                                                                       \
        }                                                                                                     \
    } while (0)

int main() {
    long plans = 0, split = 0, none = 0;
    const int Ts[] = {65, 100, 128, 129, 201, 256, 257, 384, 1000, 1024, 4096, 100000};
    const int64_t Ns[] = {1, 255, 256, 257, 512, 3584, 8960, 18944, 18947, 152064};
    const int Gs[] = {1, 2, 3, 12, 24, 28, 70, 148, 1024};
    for (int T : Ts)
        for (int64_t N : Ns)
            for (int G : Gs)
                for (int bm : {128, 256})
                    for (int lo = 0; lo < 2; lo++)
                        for (int cus : {1, 64, 256})
                            for (int64_t part : {int64_t(0), int64_t(4) << 20, int64_t(16) << 20})
                                for (int least : {1, 3}) {
                                    const iq::GemmwPlan p = iq::gemmw_plan(T, N, G, bm, lo, cus, part, least);
                                    ++plans;
                                    if (p.us > 1e29) {  // refused: only where so many ranges do not fit
                                        ++none;
                                        CHECK(least > 1);
                                        continue;
                                    }
                                    const int64_t tiles = int64_t(p.tiles_m) * p.tiles_n;
                                    CHECK(int64_t(p.tiles_m) * bm >= T && int64_t(p.tiles_n) * 256 >= N);
                                    CHECK(p.full >= 0 && p.full <= tiles && p.full % cus == 0);
                                    CHECK(p.splits >= 1 && p.gch >= 1);
                                    CHECK(int64_t(p.splits) * p.gch >= G);       // every group
                                    CHECK(int64_t(p.splits - 1) * p.gch < G);    // no empty range
                                    if (p.splits > 1) {
                                        ++split;
                                        CHECK(p.splits * (tiles - p.full) * bm * 256 <= part);
                                    }
                                    if (least > 1 && G >= least) CHECK(p.splits >= 2);
                                }
    // rows so long that a tile's 32-bit byte offsets would wrap are refused
    for (int G : {1 << 15, 1 << 16, (1 << 17) - 1})
        for (int T : {65, 300, 1024})
            for (int64_t N : {int64_t(4096), int64_t(8192)})
                for (int bm : {128, 256}) {
                    const int lo = 0, cus = 256, least = 1;
                    const int64_t part = int64_t(16) << 20;
                    CHECK(int64_t(bm) * G * 256 < (int64_t(1) << 31) || iq::gemmw_plan(T, N, G, bm, lo, cus, part, least).us > 1e29);
                }
    std::printf("%ld plans checked, %ld split, %ld refused, %d failures\n", plans, split, none, failures);
    return failures ? 1 : 0;
}

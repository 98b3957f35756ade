// iq_plan.h -- host-only launch planning shared by the launchers and the
// CPU tests (plain C++: no HIP types, so g++ compiles it on its own).
#pragma once

#include <algorithm>
#include <cstdint>

namespace iq {

// K ranges of a gemvq launch (M in 7..32 activation rows, G 128-column
// groups, `tiles` 16-row and `t32` 32-row tiles over all matrices, `kind`
// 0 int8 / 1 int4, `cus` compute units, `part_floats` the split-K partial
// sums the workspace holds).
//   gs  groups per range;
//   S   workgroups along K (S > 1: each writes M x tiles x 16 partial sums,
//       S of them must fit part_floats);
//   L   consecutive ranges per workgroup (1: one range each; > 1 the looped
//       kernel instance, ranges of ngl groups);
//   mb  16-row activation blocks (1 or 2).
struct GqPlan {
    int gs = 0, S = 0, L = 1, ngl = 0, mb = 0, nrb = 0;
    bool ok = false;
};

inline GqPlan gemvq_plan(int64_t G, int M, int tiles, int t32, int kind, int cus, int64_t part_floats) {
    GqPlan pl;
    if (M < 7 || M > 32 || G < 1 || tiles < 1) return pl;
    pl.nrb = (t32 + 7) / 8;
    // ranges of at most ngr groups (the weights of a range are held in
    // registers: 64 per lane at one row block; the operands of 2 blocks x 4
    // groups fill 64 KiB of LDS), and enough workgroups for two per CU
    pl.mb = M <= 16 ? 1 : 2;
    const int ngr = pl.mb == 2 ? 4 : (kind == 1 ? 6 : 4);
    const int want = 2 * cus;
    int S = int((G + ngr - 1) / ngr);
    S = std::max<int>(S, std::min<int>((want + pl.nrb - 1) / pl.nrb, int(G)));
    int gs = int((G + S - 1) / S);
    S = int((G + gs - 1) / gs);
    int L = 1;
    int ngl = ngr;
    const int64_t outs = int64_t(M) * tiles * 16;  // partial sums per workgroup along K
    if (S > 1 && int64_t(S) * outs > part_floats) {
        // partial sums beyond the workspace: fewer workgroups along K, each
        // taking L consecutive ranges; when not even two sets fit, one
        // workgroup per row block takes every range and stores y directly.
        // (int8 at two row blocks loops over 2-group ranges: 110 VGPRs,
        // two workgroups per CU, against 150 with 4)
        if (kind == 0 && pl.mb == 2) ngl = 2;
        const int R = int((G + ngl - 1) / ngl);
        gs = int((G + R - 1) / R);
        const int64_t fit = std::max<int64_t>(part_floats / outs, 1);
        L = int((R + fit - 1) / fit);
        S = (R + L - 1) / L;
    }
    pl.gs = gs;
    pl.S = S;
    pl.L = L;
    pl.ngl = ngl;
    pl.ok = S == 1 || int64_t(S) * outs <= part_floats;
    return pl;
}

// Tiles of a wide-tile prefill GEMM (iq_gemmw.hip; T x N outputs, G
// 128-column groups, bm x 256 tiles, one workgroup per CU): whole tiles for
// as many full rounds of the CUs as there are, and the rest over `splits`
// ranges of gch groups, the number with the least estimated time of rounds x
// groups and of the range sums' way through memory (each range of a tile
// writes bm x 256 sums; all must fit part_floats).  least: the fewest ranges
// to take (> 1: every tile is split).  us: the estimate; above 1e29 when no
// plan fits.  The times per group and round are measured: bf16 at bm = 256 /
// 128, 16384 x 4096 at T = 1024 143 / 195 us, fp32 246 us (one, two and two
// rounds of 32 groups); the sums cost 8 bytes a float at 9 TB/s (they stay
// in the last-level cache) and a launch.  Splitting only the last, partly
// filled round: 7B gate at T = 1024, bf16 222 -> 171 us, fp32 307 -> 296.
struct GemmwPlan {
    int bm = 0, tiles_m = 0, tiles_n = 0, full = 0, splits = 1, gch = 0;
    double us = 1e30;
};

inline GemmwPlan gemmw_plan(int64_t T, int64_t N, int64_t G, int bm, bool lo, int cus, int64_t part_floats, int least) {
    GemmwPlan pl;
    pl.bm = bm;
    pl.tiles_m = int((T + bm - 1) / bm);
    pl.tiles_n = int((N + 255) / 256);
    const int64_t tiles = int64_t(pl.tiles_m) * pl.tiles_n;
    // (a tile's byte offsets are 32 bits wide: 256 rows of 2 K bytes stay
    // below 2^31 for K < 2^22)
    if (tiles > (1 << 24) || G >= (1 << 15)) return pl;
    pl.full = least > 1 ? 0 : int(tiles / cus * cus);
    pl.gch = int(G);
    const int64_t tail = tiles - pl.full;
    const double group_us = bm == 256 ? 4.3 : lo ? 3.7 : 2.9;
    const double full_us = 8.0 + double(pl.full / cus) * double(G) * group_us;
    double best = tail == 0 ? 0.0 : 1e30;
    for (int S = least; tail > 0 && S <= 16 && S <= G; S++) {
        const int gch = int((G + S - 1) / S), n = int((G + gch - 1) / gch);
        const int64_t floats = n * tail * bm * 256;
        if (n > 1 && floats > part_floats) break;
        const double us = double((tail * n + cus - 1) / cus) * gch * group_us +
                          (n > 1 ? 5.0 + double(floats) * 8 / 9e6 : 0.0);
        if (us < best) {
            best = us;
            pl.splits = n;
            pl.gch = gch;
        }
    }
    pl.us = full_us + best;
    return pl;
}

}  // namespace iq

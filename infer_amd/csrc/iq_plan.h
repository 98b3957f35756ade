// iq_plan.h -- host-only launch planning shared by the launchers and the
// CPU tests (plain C++: no HIP types, so g++ compiles it on its own).
#pragma once

#include <algorithm>
#include <cstdint>

namespace iq {

constexpr int kMaxRowsGemv = 32;  // GpuBatch::kMaxRows (kernels/batch_gpu.h:80)

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

// The rows that take the 1-row kernel: 1..4 always; 5..8 rows (two blocks of 4, the second converted after
// the first is multiplied) only on narrow launches, measured at 7B: o (224
// tiles) 10.1 -> 9.2 us at 8 rows and q|k|v (288) 12.2 -> 10.5 at 5, but
// q|k|v 12.2 -> 13.1 at 8 rows and gate|up 35 -> 41 / 53 us at 5 / 8.
inline bool gemv1_rows_preferred(int M, int tiles, int64_t G, int cus) {
    if (M <= 4) return true;
    if (M > 8) return false;
    // short rows convert fast: 1.5B gate (G = 12, 560 tiles) at 7 / 8 rows
    // 11.7 -> 10.1 / 11.8 -> 10.7 us (int8)
    return tiles <= cus || (tiles < 4 * cus && (M <= 6 || G <= 16));
}

// gemvw's ranges and workgroups for M rows, `units` 16-row tiles (or SwiGLU
// pairs of them): S ranges of gs groups, nw waves of ng groups a workgroup,
// nrb workgroups a range.  ok: G is whole sets of ng groups.
struct GwPlan {
    int ng = 0, S = 0, gs = 0, nw = 0, nrb = 0;
    bool ok = false;
};

inline GwPlan gemvw_plan(int64_t G, int M, int units, int cus) {
    GwPlan pl;
    // groups a wave: 4 (2 from 17 rows: their operands fill the registers),
    // or 2 where G leaves a remainder and on short rows, whose few waves
    // would otherwise leave half the CU's registers unused (1.5B gate|up, G =
    // 12, at 16 rows int4 / int8 14.0 / 15.0 -> 10.9 / 11.6 us, 5 rows 10.7
    // / 12.1 -> 10.3 / 10.2); whole sets only
    pl.ng = M <= 16 && G % 4 == 0 && G > 16 ? 4 : 2;
    if (M < 5 || M > kMaxRowsGemv || G % pl.ng) return pl;
    pl.S = int((G + 8 * pl.ng - 1) / (8 * pl.ng));
    pl.gs = int((G + pl.S - 1) / pl.S);
    pl.gs = (pl.gs + pl.ng - 1) / pl.ng * pl.ng;
    pl.S = int((G + pl.gs - 1) / pl.gs);
    pl.nw = pl.gs / pl.ng;
    const int slots = cus * (8 / pl.nw);
    pl.nrb = std::min(units, std::max(1, slots / pl.S));
    // (one or two tiles a workgroup: two each, so that no CU waits for a
    // second workgroup)
    if (units < 2 * pl.nrb && units > pl.nrb) pl.nrb = (units + 1) / 2;
    pl.ok = true;
    return pl;
}

// gemvw or the other kernels (both measured in a graph, us, others -> gemvw):
// 17..32 rows from 64 tiles on (7B k 512 x 3584 at 17 rows 11.2 kept against
// 11.4; 1024 x 7168 16.9 -> 12.6); 9..16 rows on long rows (1.5B down, G =
// 70, int8 20.9 -> 11.0, int4 15.2 -> 10.2) or where tiles x groups fill the
// card (7B q|k|v, 288 x 28, 12.3 -> 11.4; o, 224 x 28, int4 9.7 kept against
// 10.4, int8 11.9 -> 11.1; 7168 x 1024, 448 x 8, 7.6 kept against 8.9: the
// two lines lie closely about o's 6272, between the two other shapes, and
// nothing nearer was measured); 5..8 rows wherever the 1-row kernel's exact
// integer sums do not serve (on those narrow calls, where gemvw would be up
// to 25 % faster at 8 rows, its error is 1.2 to 1.4 times theirs).
inline bool gemvw_preferred(int M, int tiles, int64_t K, int kind, int cus) {
    const int64_t G = K / 128;
    if (M < 5 || M > kMaxRowsGemv || K % 128 || G % 2) return false;
    if (M > 16) return tiles >= 64;
    if (M > 8) return G >= 48 || tiles * G >= (kind == 1 ? 6400 : 6000);
    return tiles >= 1024 || G >= 128 || !gemv1_rows_preferred(M, tiles, G, cus);
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
// rounds of 32 groups; int8 codes, and int4 takes up to a quarter longer in
// bf16, 7B gate's product 160 / 199 us, which the estimate leaves out); the
// sums cost 8 bytes a float at 9 TB/s (they stay in the last-level cache) and
// a launch.  Splitting only the last, partly filled round: 7B gate at T =
// 1024, bf16 222 -> 171 us, fp32 307 -> 296.
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

// Rows of gemm_kernel's tiles (16-byte loads; bf16a: bf16 activations on its
// aligned loads).
// 64-row tiles for short T (less MFMA work on padding rows, more tiles):
// 7B int8, fp32 activations, gate 18944 x 3584 at T = 33 / 64 / 128 /
// 256: 115 / 113 / 137 / 202 -> 55 / 58 / 97 / 139 us; down 3584 x
// 18944 at T = 64 / 256: 115 / 186 -> 58 / 170 us, but at T = 128 (a
// narrow matrix, already split over K) 93 -> 103: kept at 128 rows there
// 256-row tiles (8 waves) for long bf16 prefills of narrow int4
// matrices: each dequantised weight tile (nibble unpack + zero point,
// the costlier conversion) feeds twice the MFMAs.  7B at T = 1024 with
// 256 / 128 rows: int4 down 259 / 275 us, int4 gate|up 235 / 208 us,
// int8 down 269 / 249 us (one 8-wave workgroup per CU leaves the step
// barriers uncovered, which costs more than the conversion saves on a
// wide matrix or with int8's cheaper conversion).
inline int gemm_rows(int64_t T, int64_t N, int kind, bool bf16a) {
    if (T <= 64 || (T > 128 && T <= 256) || (T <= 128 && N >= 8192)) return 64;
    return bf16a && T >= 512 && kind == 1 && N < 8192 ? 256 : 128;
}

// Rows of the fp16 operand path's tiles (gemmh_kernel).
// 64 x 128 tiles on 4 waves, two workgroups per CU (a 4-wave workgroup
// of 128 rows, whose hi + lo operand buffers fill the LDS, runs alone
// on its CU: 7B int8 at T = 128 / 512 / 1024, down 3584 x 18944 99 /
// 334 / 684 -> 66 / 212 / 433 us, gate 18944 x 3584 266 / 440 -> 201 /
// 393 us at 512 / 1024, o 3584 x 3584 at 1024 142 -> 93 us).  From T =
// 512, int4 and rows of K >= 2048 take 128 x 128 tiles on 8 waves, each
// converted weight tile feeding twice the rows: 7B int4 at T = 1024 /
// 2048 down 426 / 936 -> 378 / 782 us, gate 389 / 801 -> 354 / 721 us,
// int8 gate 402 -> 381 us at 1024 (1.5B int8 gate 8960 x 1536: 110 ->
// 116 us, kept at 64 rows).
inline int gemmh_rows(int64_t T, int64_t K, int kind) { return T >= 512 && (kind == 1 || K >= 2048) ? 128 : 64; }

// Whether gemm_kernel splits fp32 activations itself: past 32 rows on whole
// 128-column groups the fp16 operand path (22 significant bits against the
// 24 of three bf16 terms at 1.5x the MFMAs, and faster: 7B at T = 1024, gate
// 18944 x 3584 int4 648 -> 440 us, down 1053 -> 681 us); up to 32 rows the
// three-term split inside gemm_kernel, whose single launch beats the
// preparation launch on the narrower matrices left here (1.5B at 32 rows: o
// 1536 x 1536 16.9 -> 11.6 us, down 1536 x 8960 25.4 -> 21.8; 7B o 22.9
// either way), and so up to 64 rows on matrices of at most 2^24 weights (T =
// 64: 1.5B o 15.6 -> 10.2, down 24.1 -> 19.7, 7B o 23.7 -> 21.4 us; 7B gate
// 44.8 against 64.7) and up to 256 rows on matrices of at most 2^22 (T =
// 96..256: 7B k 512 x 3584 18.0..22.4 -> 13.3..14.6 us, 1.5B o 23.2..25.1 ->
// 17.7..22.4), at any T on matrices of at most 2^19 (1.5B k 256 x 1536 at T
// = 257 / 512 / 2048: 17.3 / 20.7 / 34.0 -> 12.7 / 12.4 / 25.9 us)
inline bool gemm_splits_x(int64_t T, int64_t N, int64_t K) {
    const int64_t nk = N * K;
    return T <= 32 || (T <= 64 && nk <= (int64_t(1) << 24)) || (T <= 256 && nk <= (int64_t(1) << 22)) ||
           nk <= (int64_t(1) << 19);
}

// Few output tiles (short T): split K into ranges of whole 128-column groups
// so that the tiles x ranges fill the workgroup slots of the CUs (per_cu
// resident workgroups of the instance per CU) in one round, the range sums
// added by gemm_reduce_kernel; needs room for the sums.  Rounding the range
// count down rather than up keeps a second, mostly idle round of workgroups
// off the critical path (7B down 3584 x 18944 at T = 80 / 200, fp32 activations: 76.8 / 140.6 -> 60.7 / 111.0
// us; bf16 activations 50.1 / 94.9 -> 36.6 / 69.4 us; 7B gate 18944 x 3584
// with bf16 activations at T = 17..48, on the three-term kernel's one
// workgroup per CU: 29.5..32.6 -> 24.1..27.0 us).  The exception: tiles
// that fill only half to two thirds of one round, on rows of at least 24
// groups, take 3 ranges (two full rounds of shorter workgroups; 7B gate at
// T = 65 / 96 / 128, int8, fp32 activations 78.0 / 72.9 / 73.3 -> 66.4 /
// 64.9 / 68.7 us, bf16 activations 49.6 / 49.7 / 50.2 -> 41.8 / 43.8 /
// 46.5 us, int4 8-16 % faster; 1.5B gate 8960 x 1536, 12 groups, at T =
// 256 lost 38.2 -> 44.5 us), and so do tiles that fill one round up to 2.5
// rounds (7B gate at T = 256, int8 / int4: fp32 activations 125.9 / 119.8
// -> 116.3 / 107.5 us, bf16 84.9 / 95.9 -> 81.8 / 88.9 us; wider ones
// overrun the partial sums).  part_floats: the workspace's partial-sum
// capacity.
inline int pick_splits(int tiles, int slots, int64_t G, int64_t T, int64_t N, int64_t part_floats) {
    if (G < 2) return 1;
    if (tiles >= slots) {
        if (2 * tiles < 5 * slots && G >= 24 && 3 * T * N <= part_floats) return 3;
        return 1;
    }
    int S = slots / tiles;
    S = S > 16 ? 16 : S;
    while (S > 1 && int64_t(S) * T * N > part_floats) S--;
    if (S == 1 && 3 * tiles <= 2 * slots && G >= 24 && 3 * T * N <= part_floats) S = 3;
    return S;
}

// S ranges of whole groups over G groups: the groups of a range, and the
// ranges these make.
struct KRanges {
    int64_t gch;
    int splits;
};
inline KRanges k_ranges(int S, int64_t G) {
    if (S < 2) return {G, 1};
    const int64_t gch = (G + S - 1) / S;
    return {gch, int((G + gch - 1) / gch)};
}

// Estimated time of tiles x S K ranges on the narrow tiles, workgroups of
// which per_cu share a CU, group_us a group and round (measured: 7B gate
// 18944 x 3584, T = 201 and 384..1024), plus the range sums' way through
// memory: what the wide tiles' estimate is compared with (GemmwPlan).  Both
// sides at the line, fp32 int8: 7B gate at T = 160 / 201 86 / 120 -> 86
// (kept) / 105 us, o 3584 x 3584 at T = 384 / 512 47 / 55 -> 46 / 52, 1.5B
// gate 8960 x 1536 at T = 384 / 512 45 (kept) / 66 -> 44 / 57; bf16: 7B gate
// at T = 300 / 384 80 / 83 (kept) against 88 / 112 on the wide tiles, at T =
// 450 133 -> 113.
inline double narrow_us(int tiles, int per_cu, int S, int64_t G, int64_t T, int64_t N, double group_us, int cus) {
    const int slots = per_cu * cus;
    const int64_t gch = (G + S - 1) / S;
    return 4.0 + double((int64_t(tiles) * S + slots - 1) / slots) * double(gch) * group_us +
           (S > 1 ? 5.0 + double(S) * double(T) * double(N) * 8 / 9e6 : 0.0);
}

// The wide tiles' plan for a prefill GEMM that may take them (whole groups,
// 16-byte aligned operands; lo: fp32 activations as fp16 hi + lo), or one
// with us > 1e29 where the narrow tiles' estimate is the lower.
inline GemmwPlan gemmw_choose(int64_t T, int64_t N, int64_t K, int kind, bool lo, int cus, int64_t part_floats) {
    const int64_t G = K / 128;
    if (T <= 64) return GemmwPlan{};
    double narrow;
    if (lo) {
        const int bm = gemmh_rows(T, K, kind), per_cu = bm == 128 ? 1 : 2;
        const int tiles = int((T + bm - 1) / bm) * int((N + 127) / 128);
        narrow = narrow_us(tiles, per_cu, k_ranges(pick_splits(tiles, per_cu * cus, G, T, N, part_floats), G).splits, G, T,
                           N, bm == 128 ? (kind == 1 ? 2.45 : 2.65) : (kind == 1 ? 2.05 : 2.4), cus);
    } else {
        const int bm = gemm_rows(T, N, kind, true), rows = bm == 256 ? 128 : bm;
        const int tiles = int((T + rows - 1) / rows) * int((N + 127) / 128);
        narrow = narrow_us(tiles, 2, pick_splits(tiles, 2 * cus, G, T, N, part_floats), G, T, N, bm == 64 ? 1.9 : 2.8, cus);
    }
    // (bf16 rows of at least 24 groups at T <= 256 keep the three or more
    // ranges, and with them the shorter sums, that the narrow tiles have)
    const int least = !lo && T <= 256 && G >= 24 ? 3 : 1;
    GemmwPlan pl = gemmw_plan(T, N, G, 128, lo, cus, part_floats, least);
    if (!lo) {
        const GemmwPlan p8 = gemmw_plan(T, N, G, 256, lo, cus, part_floats, least);
        if (p8.us < pl.us) pl = p8;
    }
    // (the estimates are good to some percent: 5 % in doubt for what is there)
    return pl.us > 0.95 * narrow ? GemmwPlan{} : pl;
}

}  // namespace iq

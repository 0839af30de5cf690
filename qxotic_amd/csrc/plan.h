// Which kernel of a family takes a call and how it splits k: plain arithmetic on the call's sizes, shared by the launchers,
// by the sizing of their scratch and by the tests (compiles without HIP).
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "dtype.h"

namespace jamhip {

inline int up_div(int a, int b) { return (a + b - 1) / b; }

// Bytes from one row of a device copy of dense weights to the next. Rows start on 256 bytes, so 16-byte aligned for vector loads;
// from 4096 bytes on the pitch is an odd multiple, so that rows of a power-of-two length do not all start on one memory
// channel (one token, us, even against odd: F16 8192x2048 9.6 / 8.1, 32000x2048 26.8 / 23.5, 4096x4096 9.7 / 8.8, 14336x4096 23.5 /
// 22.5, F32 32000x1024 26.1 / 22.0). Shorter rows share DRAM pages that the gap would break up (F16 32000x1024 n = 64 33.3 /
// 37.7, 4096x256 n = 4 4.97 / 5.33), and would pay for it with up to half as much memory again; from there on it is 1/16 at most.
constexpr int64_t dense_row_pitch(int64_t row_bytes) {
    const int64_t units = (row_bytes + 255) / 256;
    return (units >= 16 ? units | 1 : units) * 256;
}

// K slices of a matrix-core GEMM: ns of them, `per` K units each (0 when whole).
struct Split {
    int ns, per;
};

// K slices for a grid of `total` workgroups: enough for about two workgroups per CU, whole units each.
inline Split split_plan(int total, int units) {
    int want = total >= 384 ? 1 : up_div(512, total);
    want = want < units ? want : units;
    const int per = want > 1 ? up_div(units, want) : 0;
    return {want > 1 ? up_div(units, per) : 1, per};
}

// Workgroups of two resident per CU take about the same CU time whether a CU holds one or two, so a call
// takes ceil(tiles per CU) tile times: Q4_K 14336x4096 at n = 448, 512 and 576 (784, 896 and 1008 tiles)
// all ran 128 us. Each XCD takes a contiguous run of T8 = ceil(tiles / 8) tiles over its CUs; when that
// leaves r <= CUs / 2 tiles for a last partial round, those r tiles run as 2r half tiles (32 tokens) instead,
// one per CU. Returns r, or 0 for no split.
inline int tail_tiles(int total, int cus) {
    if (cus < 8) return 0;   // not primed: no split
    const int cu8 = cus / 8, r = up_div(total, 8) % cu8;
    return r > 0 && 2 * r <= cu8 ? r : 0;
}

// Half tiles that the fullest CU computes, for `total` tiles times `ns` K slices.
inline int cu_half_tiles(int total, int ns, int cus, bool tail) {
    const int cu8 = cus < 8 ? 32 : cus / 8, t8 = up_div(total, 8) * ns, r = t8 % cu8;
    return 2 * (t8 / cu8) + (r == 0 ? 0 : tail && 2 * r <= cu8 ? 1 : 2);
}

// The K-quants past 64 tokens: kq_wide_kernel (128 x 128 tiles), or kq_gemm_kernel (128 x 64). Both leave CUs idle in their
// last round, at different sizes, so neither is the faster one from some size on; the rule compares what the fullest CU has
// to do, in super-block times of a 128 x 64 tile. A wide tile takes 1.6 of them (one half of it padding or not), its longer
// start and end 3, and each million floats of split-K partials 0.3. Both kernels with prep and reduce, in us:
//   Q4_K 14336x4096 n = 512 (448 wide tiles, 2 rounds, against 3.5) 103 / 111; n = 576 (560, 3 against 4) 137 / 120;
//   n = 260 (336, 2 against 2.5) 92 / 83; n = 2048 366 / 433; 28672x4096 n = 260 161 / 134; 12288x4096 n = 384 93 / 87;
//   16384x1024 n = 65 (1 super-block per slice) 27.8 / 22.5; Q5_K 14336x4096 n = 576 152 / 140; Q6_K 4096x14336 n = 512
//   (128 tiles, 4 slices for 2) 153 / 168, n = 129 76 / 72; 12288x4096 n = 260 107 / 87; 16384x1024 n = 129 (2 slices for 1) 1.4 : 1.
// Over 867 such points (14 shapes, 65 to 2048 tokens) no call that goes to the wide kernel was over 1.1% behind the other.
// Two exceptions are in it: Q4_K, the lightest to decode, is not split where kq_gemm_kernel is whole, nor whole where the
// scratch left no room to split (4096x14336 n = 1024, 256 workgroups, 242 / 227), and three blocks of 64 tokens, padded to
// four, are not split finer past 4 slices (Q6_K 4096x14336 n = 129, above, 8 slices for 6).
// kq_wide_kernel addresses a super-block's codes and the next one's first by 32-bit offsets: up to 11 blocks of 64 bytes a
// token, which pass 2^32 at 6.1 million.
constexpr int WIDE_MAX_TOKENS = 1 << 22;
struct WidePlan {
    bool wide;
    Split k;
};
inline WidePlan wide_plan(int dt, int k, int m, int n, int cus, size_t act_bytes) {
    if ((dt != Q4_K && dt != Q5_K && dt != Q6_K) || n <= 64) return {false, {1, 0}};
    const int NP = up_div(n, 64) * 64, nsb = up_div(k, 256), rows = up_div(m, 128);
    if (NP > WIDE_MAX_TOKENS) return {false, {1, 0}};
    const int total = rows * up_div(NP, 128), ototal = rows * (NP / 64);
    const Split o = split_plan(ototal, nsb);
    // about two workgroups per CU
    int want = total >= 320 ? 1 : (512 + total / 2) / total;
    want = want < nsb ? want : nsb;
    // scratch past what the other kernel's slices take must leave every allocation-free call inside its 64 MiB
    while (want > o.ns && act_bytes + (size_t) want * n * m * 4 > ((size_t) 60 << 20)) want--;
    Split s{1, 0};
    if (want > 1) s.per = up_div(nsb, want), s.ns = up_div(nsb, s.per);
    const bool split = s.ns > 1, osplit = o.ns > 1;
    if (dt == Q4_K && (split ? !osplit : total < 320)) return {false, {1, 0}};
    if (NP == 192 && s.ns > o.ns && s.ns > 4) return {false, {1, 0}};
    const double part = 0.3e-6 * n * m;
    const double wide = 1.6 * (split ? s.per : nsb) * cu_half_tiles(total, s.ns, cus, false) / 2 + (split ? s.ns * part : 0) + 3;
    const double other = (double) (osplit ? o.per : nsb) * cu_half_tiles(ototal, o.ns, cus, !osplit) / 2 + (osplit ? o.ns * part : 0);
    return {wide < other, s};
}

// MXFP4 (mx4.hip): waves of 64 rows (256-row workgroups, k whole) once those give each CU one, or at k <= 4096, where a
// whole k is short, once they give every third CU one; else waves of 32 rows with the K split of the other types.
// 64 against 32 rows: 14336x4096 n = 320 55.7 / 67.2 us (280 workgroups), n = 512 72.8 / 80.1, n = 128 36.5 / 38.8 (112),
// 5760x2880 n = 256 27.5 / 32.0 (92), n = 512 37.9 / 41.8; but 14336x4096 n = 64 34.4 / 24.7 (56), 4096x14336 n = 512 111 /
// 84 (128). A whole k of 64-row waves split like the others measures as the 32-row waves do.
inline int mx4_row_tiles(int m, int k, int ncb) { return m >= 512 && up_div(m, 256) * ncb >= (k <= 4096 ? 88 : 256) ? 2 : 1; }
struct Mx4Plan {
    int rt, tiles;   // row tiles per wave, workgroup tiles
    Split k;
};
inline Mx4Plan mx4_plan(int m, int k, int n) {
    const int ncb = up_div(n, 64), rt = mx4_row_tiles(m, k, ncb), tiles = up_div(m, 128 * rt) * ncb;
    return {rt, tiles, rt == 1 ? split_plan(tiles, up_div(k, 256)) : Split{1, 0}};
}

// The staged dense GEMMs (F16, and BF16 with rounded activations): dense_mma_kernel's 128 x 64 tiles, two workgroups per CU, or
// dense_big_kernel's 256 x 128, one per CU, over the same K slices of `units` stages of 64. As for the K-quants, what the
// fullest CU computes decides, in stages of a 128 x 64 tile, of which a CU overlaps two and which ends with 2 more (BF16 0.5): a
// stage of a big tile takes 1.7 of them (1.3), its start and end, which nothing on its CU overlaps, 5 (4), and the call 5 (8).
// Both kernels over the same prep in 320 F16 and 320 BF16 calls (34 shapes from 32x2880 to 60000x256, 65 to 1024 tokens),
// in us, big first:
//   F16 14336x4096 n = 512 121 / 229, n = 65 (3 slices) 53 / 85; 6144x4096 n = 80 31 / 41; 8192x4096 n = 1024 132 / 229;
//   4096x14336 n = 129 91 / 142; but 257x4096 n = 128 (22 slices of 3 stages) 76 / 42, 256x4096 n = 512 37 / 27,
//   1000x1024 n = 256 26 / 24, 4096x128 n = 512 25 / 23, 32x2880 n = 512 36 / 27; BF16 256x4096 n = 512 33 / 24, 18910x192
//   n = 881 61 / 52.
// One call that the rule gives to the big tiles is 2% slower for it (F16 4096x4096 n = 512 62.4 / 61.1), the others no more than
// 1.3%. Up to 64 tokens half of a big tile is padding and nothing is gained (F16 14336x4096 n = 16 58.2 / 58.2, BF16 n = 64
// 55.4 / 53.1).
inline bool dense_big(int dt, int units, int m, int n, Split s, int cus) {
    if (n <= 64) return false;
    const int per = s.ns > 1 ? s.per : units, big = cu_half_tiles(up_div(m, 256) * up_div(n, 128), s.ns, cus, false) / 2,
              other = cu_half_tiles(up_div(m, 128) * up_div(n, 64), s.ns, cus, false) / 2;
    return dt == F16 ? big * (1.7 * per + 5) + 5 < other * (per + 2.0) : big * (1.3 * per + 4) + 8 < other * (per + 0.5);
}

// dense_prep_kernel's grid: x over groups of 8 tokens, y over runs of their rows (of Kp elements), about two workgroups per CU,
// each with at least one pass of 64 runs. Workgroups go to the XCDs in turn, so past 8 groups x is a multiple of 8: a group's
// runs, each of which looks through the whole rows for the largest |x|, then share one L2. With 59 groups their rows went
// through all eight (F16 k = 14336 n = 469 72 -> 49 us with the product, n = 1000 85 -> 63; k = 4096 n = 136 30.3 -> 28.4).
struct PrepGrid {
    int x, y;
};
inline PrepGrid dense_prep_grid(int n, int Kp) {
    const int groups = up_div(n, 8), most = up_div(Kp / 8, 64), want = up_div(512, groups);
    return {groups > 8 ? up_div(groups, 8) * 8 : groups, want < most ? want : most};
}

// Which form of the dense activation prep: a workgroup per token (true), or 8 tokens per workgroup, the row cut into runs. The
// first reads its row in whole lines and finds its largest |x| (F16) in one pass; the second fills the CUs once rows are long
// or tokens many. By row length and tokens, measured apart from the tile form (us with the product, first form against second):
// F16 k = 512 n = 271 17.5 / 18.0; k = 1024 n = 9 12.6 / 13.1, n = 128 18.8 / 19.3, n = 512 23.4 / 23.1; k = 2000 n = 9 16.4 /
// 17.0, n = 300 21.9 / 21.0; k = 2048 n = 256 21.8 / 21.1; k = 4096 n = 9 25.4 / 24.5, n = 64 33.5 / 31.2; k = 14336 n = 9
// 86 / 73; BF16 (no largest |x|) k = 2000 n = 64 18.2 / 18.3, n = 512 19.5 / 18.5; k = 2048 n = 9 14.9 / 15.3; k = 4096 n = 64
// 29.2 / 28.6; k = 14336 n = 64 76 / 73.
inline bool dense_prep_few(int dt, int k, int n) { return n <= (k <= 1024 ? 320 : 256) && k <= (dt == F16 ? 2047 : 2048); }

// dense_tile_kernel's tile: 32 x 32 (true) halves the bytes read per product and takes over once such tiles give most CUs one,
// but up to 16 tokens half of it is padding. 16 x 16 against 32 x 32, us: F32 512x2880 n = 512 (256 tiles of 32) 41.4 / 24.6,
// 2048x4096 n = 96 (192) 44.5 / 32.7; 256x4096 n = 512 (128) 30.6 / 32.1, 2048x4096 n = 64 (128) 30.8 / 32.2; 14336x4096
// n = 5 49 / 71, n = 16 62 / 71, n = 17 (448) 101 / 71, 32000x2048 n = 9 54 / 68.
inline bool dense_tile32(int m, int n) { return n > 16 && (int64_t) up_div(m, 32) * up_div(n, 32) >= 192; }

}  // namespace jamhip

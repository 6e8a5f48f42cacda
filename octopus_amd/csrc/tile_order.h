// The GEMMs' workgroup -> tile order, as constexpr functions of plain integers: hipcc compiles them for the GPU
// (constexpr functions are callable from device code), and g++ for the CPU check of the order
// (tests/plan_check.cpp, under -fsanitize=address,undefined).
//
// Block -> (mt, nt). Blocks run on XCD b % 8. The first 8 * floor(M-tiles / 8) M-tiles are dealt to the XCDs
// round-robin (XCD x owns mt = x, x + 8, ...), and each XCD walks its own in groups of group_m across all N-tiles, so
// the ~32 workgroups resident on an XCD run 4 M-tiles x 8 N-tiles and share A and B K-slices in its L2, while the 8
// XCDs sweep the N-tiles in step (at 114,688 hidden rows, 0.59 GB, more than the 256 MB Infinity Cache, XCDs out of
// step made the forward 6% slower). The tiles of the last M-tiles % 8 M-tiles are cut into 8 contiguous segments of
// equal length (+-1), one per XCD, so every XCD holds the same number of tiles whatever the shape (whole M-tile rows
// for those too gave an XCD with one more row a whole extra round: 99 M-tiles x 10 N-tiles ran 5 rounds of 32 tiles on
// three XCDs against 4 on the others). Per XCD that is floor(M / 8) N + ceil((M % 8) N / 8) = ceil(M N / 8) tiles.
// A device-side row count that bounds M or N shrinks the tile grid (read once per block), so the idle blocks all come
// after the working ones instead of between them: interleaved idle blocks retire instantly and stagger the working
// workgroups at every group start, which breaks their L2 sharing. The grid is 8 * ceil(bound-free tiles / 8); blocks
// past their XCD's tiles return false.
#pragma once

#include <stdint.h>

namespace octo_tiles {

// Workgroups of the one-shot grid of mtiles x ntiles tiles: 8 ceil(tiles / 8).
constexpr int64_t tile_grid(int64_t mtiles, int64_t ntiles) { return 8 * ((mtiles * ntiles + 7) / 8); }

// Tiles XCD x holds in the order below.
constexpr int64_t xcd_tiles(int x, int64_t mtiles, int64_t ntiles) {
  const int64_t T = (mtiles % 8) * ntiles;
  return (mtiles / 8) * ntiles + (x + 1) * T / 8 - x * T / 8;
}

// XCD x's k-th tile (mt, nt) of an mtiles x ntiles grid walked in groups of group_m M-tiles; false past its tiles. In
// 32-bit integers (a grid has fewer than 2^31 blocks): every workgroup works this out before its first load, and the
// three divisions are some 400 instructions in 64 bits.
constexpr bool tile_at(int group_m, int x, int k, int mtiles, int ntiles, int &mt, int &nt) {
  const int mfull = mtiles / 8;  // M-tiles every XCD owns: x, x + 8, ..., x + 8 (mfull - 1)
  const int main = mfull * ntiles;
  if (k < main) {
    const unsigned span = (unsigned)(group_m * ntiles);
    const int gid = (int)((unsigned)k / span);
    const int first = gid * group_m;
    const unsigned gsize = (unsigned)((mfull - first) < group_m ? (mfull - first) : group_m);
    const unsigned local = (unsigned)k - (unsigned)gid * span, q = local / gsize;
    mt = x + 8 * (first + (int)(local - q * gsize));
    nt = (int)q;
    return true;
  }
  // the last r M-tiles, M fastest, cut in 8
  const unsigned r = (unsigned)(mtiles - 8 * mfull), T = r * (unsigned)ntiles;
  const unsigned L = (unsigned)x * T / 8 + (unsigned)(k - main);
  if (L >= (unsigned)(x + 1) * T / 8) return false;
  const unsigned q = L / r;
  mt = 8 * mfull + (int)(L - q * r);
  nt = (int)q;
  return true;
}

// ---- split K (grad_h) ----------------------------------------------------------------------------------------
//
// grad_h = dz . W contracts over the vocabulary: few tiles (rows / 256 x d / 256), each long (V / 64 stages). With
// fewer tiles than CUs the long tiles set the time: 225 scored rows at d 2560, V 151,936 are 10 tiles of 2,374 stages,
// 3.0 ms on 10 CUs while grad_W's 5,940 tiles of 4 stages keep the others busy for 0.3. So a tile's K is cut into S
// runs of whole stages, each a workgroup of its own that leaves an fp32 partial tile, which a small kernel sums in run
// order.
//
// k_splits: S for `tiles` tiles of nk stages. A run keeps at least kSplitStages stages (a partial tile costs about
// kSplitCost stages of time to write and sum: 256 KB each way at 5 TB/s over 256 CUs, against 1.25 us a stage), and
// tiles x S stays within cap, the partial tiles the workspace holds.
//   beside grad_W (alone = false): the short tiles fill any CU the long ones leave, so a run need only be no longer
//     than a CU's share of both products, tiles x nk / 128 stages: S = ceil(144 / tiles), none from 144 tiles on. us a
//     step and its backward, unsplit and in two runs, at d 2560, V 151,936: 120 tiles 6,044 and 6,019, 130 tiles 6,720
//     and 6,518, 140 tiles 7,076 and 6,951; 112 tiles at d 4096, V 128,256 5,001 and 4,905.
//   alone: whole rounds of the 256 CUs count, r of them with S = floor(256 r / tiles) runs, each run nk / S stages and
//     its partial tile: the cheapest of r = 1 .. 4 and of no split (120 tiles: r = 1, S = 2, half of the time; 200
//     tiles: r = 4, S = 5, 0.83 of it; 250 tiles: none).
// 32-bit integers: every block of a launch works these out.
constexpr int kSplitStages = 16, kSplitCost = 21, kCus = 256;
constexpr int kSplitItemsMax = 4 * kCus;
constexpr int k_splits(int tiles, int nk, bool alone, int cap) {
  if (tiles <= 0 || cap <= tiles) return 1;
  int most = nk / kSplitStages;
  if (most > cap / tiles) most = cap / tiles;
  if (most < 2) return 1;
  if (!alone) {
    const int s = (144 + tiles - 1) / tiles;
    return s < most ? s : most;
  }
  int best = 1, cost = ((tiles + kCus - 1) / kCus) * nk;
  for (int r = 1; r <= 4; ++r) {
    int s = kCus * r / tiles;
    if (s > most) s = most;
    if (s < 2) continue;
    const int c = ((tiles * s + kCus - 1) / kCus) * ((nk + s - 1) / s + kSplitCost);
    if (c < cost) {
      cost = c;
      best = s;
    }
  }
  return best;
}

// XCD x's k-th of the S x mtiles x ntiles runs: run-major (the tiles of one run of K read the same rows of both
// operands), M fastest within a run, cut into 8 contiguous segments; false past its segment.
constexpr bool split_item_at(int x, int k, int S, int mtiles, int ntiles, int &s, int &mt, int &nt) {
  const int t = mtiles * ntiles, T = S * t, L = x * T / 8 + k;
  if (L >= (x + 1) * T / 8) return false;
  s = L / t;
  const int p = L - s * t;
  nt = p / mtiles;
  mt = p - nt * mtiles;
  return true;
}
// First stage of run s of S over nk stages (run s ends where s + 1 begins).
constexpr int split_stage(int s, int S, int nk) { return (int)((int64_t)s * nk / S); }

// The most runs any row count up to mtiles M-tiles makes (0: none of them splits), over K of nk stages.
constexpr int split_items(int64_t mtiles, int64_t ntiles, int64_t nk, bool alone) {
  int most = 0;
  for (int64_t m = 1; m <= mtiles && m * ntiles < kSplitItemsMax; ++m) {
    const int t = (int)(m * ntiles), s = k_splits(t, (int)nk, alone, kSplitItemsMax);
    if (s > 1 && t * s > most) most = t * s;
  }
  return most;
}

}  // namespace octo_tiles

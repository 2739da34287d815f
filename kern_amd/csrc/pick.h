// Which kernel a GEMM or GEMV call launches, from its sizes alone. No HIP in here, so that the rules can be checked on the
// CPU; kern_amd/manifest.py makes the same choices for the manifest ops.
#pragma once
#include <stdint.h>

#include <algorithm>

namespace kern {

// quotients that fit 32 bits are taken there (these rules run before every launch, and 64-bit division is slow)
inline int64_t ceil_div(int64_t a, int64_t b) {
  const int64_t n = a + b - 1;
  return (n | b) >> 32 ? n / b : (int64_t)((uint32_t)n / (uint32_t)b);
}

// The walk over the weights (kern_mx_gemm_bf16_s{k / 1024}, M <= 64, k = 1024 * {1, 2, 4, 7, 8}): about 256 workgroups
// of 8 waves with at most nine half groups of 8 weight rows each.
inline int64_t walk_half_groups(int64_t m) { return std::min<int64_t>(9, ceil_div(m / 8, 256)); }

// Where the walk is taken, else the tiles below. Its waves split K, so it streams wide weights from HBM faster; its
// workgroups each read all of the activations, so more rows and narrow weights favour the tiles. Walk, tile in us:
//   M = 32, m = 9216, k = 7168 13.0, 14.4; M = 16, m = 18432, k = 8192 17.3, 19.7; M = 1, m = 4096, k = 1024 3.5, 3.7;
//   M = 16, m = 7168, k = 8192 10.6, 9.1; M = 64, m = 4096, k = 4096 10.1, 6.5; M = 40, m = 16384, k = 4096 13.5, 10.9.
// Past m = 18432 the walk needs a second round of workgroups (M = 2, m = 22528, k = 8192 24.8, 20.1) and is ahead only
// where its rounds are nearly full (0.86), at M <= 16 and k >= 7168 (M = 4, m = 33280, k = 7168 24.4, 32.9). Over 6512 shapes
// (M = 1..64, m = 2048..24576), every weight from HBM, the rule takes 0.86 of the walk's time on average and at most 3%
// more. Weights that stay in the Infinity Cache favour the tiles, whose reads it keeps (M = 64, m = 9216, k = 7168 16.8,
// 11.6, from HBM 18.4, 16.8); right behind 768 MB of writes tiles are up to 25% slower than the walk (M = 8, m = 15360,
// k = 4096).
inline bool takes_walk(int64_t M, int64_t m, int64_t k) {
  if (M > 64 || k % 1024) return false;
  const int64_t ktw = k / 1024;
  if (ktw != 1 && ktw != 2 && ktw != 4 && ktw != 7 && ktw != 8) return false;
  if (m > 18432) return M <= 16 && ktw >= 7 && m >= 15852 * ceil_div(m, 18432);
  const int64_t widest = ktw <= 2 && M <= 16 ? (ktw == 1 ? 0 : 8192)  // the widest weights that the tiles take
                         : ktw <= 4          ? 16384
                                             : 8192;
  return m > widest;
}

// The other kernels of a dense MXFP4 x MXFP8 GEMM: the small tiles (kern_mx_gemm_*_t{rows}x{weights}) and the LDS
// ring's 128 x 256 tiles. All of these accumulate K in the same order, so the choice does not show in the results.
struct SmallTile {
  int rows, weights, waves, stages;
  const char *bf16, *e4m3;  // its entries
};
#define KERN_SMALL_TILE(R, W, WAVES, STAGES) \
  {R, W, WAVES, STAGES, "kern_mx_gemm_bf16_t" #R "x" #W, "kern_mx_gemm_e4m3_t" #R "x" #W}
static const SmallTile kSmallTiles[] = {
    KERN_SMALL_TILE(16, 32, 2, 8),  KERN_SMALL_TILE(16, 64, 4, 8),  KERN_SMALL_TILE(16, 128, 8, 4),
    KERN_SMALL_TILE(32, 128, 8, 4), KERN_SMALL_TILE(48, 128, 8, 4), KERN_SMALL_TILE(80, 128, 8, 3),
    KERN_SMALL_TILE(32, 256, 8, 3), KERN_SMALL_TILE(48, 256, 8, 3), KERN_SMALL_TILE(64, 256, 8, 3),
};
#undef KERN_SMALL_TILE
// dynamic LDS of a small tile: the activation ring, then the token scales in whole KiB
inline int64_t small_tile_lds(const SmallTile& t, int64_t k) {
  return (int64_t)t.stages * t.rows * 512 + ceil_div(t.rows * (k / 512 + 1), 64) * 1024;
}
// Microseconds of a launch, fitted to both kernels over 150 shapes (M = 17..3000, N = 512..9216, K = 512..8192, graph
// replays) and corrected where 6184 more (M = 1..6144, N = 256..20480, K = 512..16384, weights from HBM and from the
// Infinity Cache) showed a bias. A tile's k group costs by its token subtiles (mt), its 16-row weight groups (n) and
// their product, its output by the product; a tile past one per CU takes a further round. Tiles that fill the chip
// are slower by a tenth, and by 40% more where K/512 is 7, 15 or 31: the weight rows of its waves then lie a power of
// two less 4 KiB apart, and their requests likely meet on the same channels (32 x 128 to 80 x 128 tiles on 180 to 256 CUs:
// 1.3, 1.6 and 1.65 times the fit, against 1.1 to 1.2 at other K).
inline double small_tile_us(const SmallTile& t, int64_t M, int64_t m, int64_t k) {
  const int64_t tiles = ceil_div(M, t.rows) * ceil_div(m, t.weights), kg = k / 512;
  const double rounds = (double)ceil_div(tiles, 256), mt = t.rows / 16, n = t.weights / 16;
  const double per_kg = -0.14 + (t.waves < 8 ? 0.2125 : 0.150) * mt + 0.0322 * n + 0.0082 * mt * n;
  const double us = 2.8 + 0.75 * (rounds - 1) + rounds * (0.045 * mt * n + (double)kg * per_kg);
  const double full = std::min(1.0, (double)tiles / 256);
  return us * (1 + 0.1 * full) * (kg >= 7 && (kg & (kg + 1)) == 0 ? 1 + 0.4 * full : 1);
}
// The ring's k group costs more as its tiles fill the chip (its clock falls). A last round that holds only tiles of a
// partial block of rows costs their share of the rows, 0.25 at least (M = 531, N = 13312, K = 10240, 52 tiles of 19 rows
// after 208 whole ones: 65 us against the 94 of two whole rounds).
inline double ring_us(int64_t M, int64_t m, int64_t k) {
  const int64_t nb = m / 256, tiles = ceil_div(M, 128) * nb, part = M % 128;
  double rounds = (double)ceil_div(tiles, 256);
  if (part && rounds > 1 && M / 128 * nb <= 256 * ((int64_t)rounds - 1))
    rounds += std::max(0.25, (double)part / 128) - 1;
  const double full = (double)tiles / 256, kg = (double)(k / 512);
  return 1.2 + rounds * (2.7 + 1.73 * kg) + full * (3.4 + 0.71 * kg);
}
// the fastest small tile for M rows by the fit (null when none takes the shape), its time in *us
inline const SmallTile* best_small_tile(int64_t M, int64_t m, int64_t k, double* us) {
  const SmallTile* best = nullptr;
  for (const SmallTile& t : kSmallTiles) {
    if (small_tile_lds(t, k) > 163840 || ceil_div(M, t.rows) > 65535) continue;
    const double u = small_tile_us(t, M, m, k);
    if (!best || u < *us) best = &t, *us = u;
  }
  return best;
}
// The rows the ring takes, a whole number of its 128-row blocks or all of them (the small tiles take the rest).
// A small tile is taken where the fit has it 10% shorter; at K > 8192 and one round of the ring its weights count at
// 4 TB/s at most (the ring's come from HBM at up to 5: M = 2, m = 33280, k = 12288 46.1 against 52.6 us). Over the 6184
// shapes the choice is within 0.5% of the fastest kernel on average, and 3.3% slower than the ring at worst; over 8462
// with m up to 160000 or k up to 65536 it is more than 3% slower than the ring or the walk at 2%, 15% at worst.
// Where the ring's last round is not full, its whole blocks of the rounds before may stay on the ring and the rest go to
// small tiles, in a launch of their own behind the ring's: taken where the fit has the two 6% shorter, 13% at K < 4096
// (there the second launch weighs more than the fit sees). Over 709 shapes with more than one round that was 97 times, 9%
// shorter on average and 0.8% longer at worst (M = 1024, N = 9216, K = 7168, 288 tiles: 70.6 -> 57.2 us, weights from HBM
// 83.0 -> 59.8; M = 2048 there, 2.25 rounds and close to the line: 126.1 -> 122.5 with its quantizer). With 5% asked for
// at every K some were 14% longer.
struct DensePlan {
  int64_t ring_rows;
  const SmallTile* tile;  // for the rest of the rows, if any
};
inline DensePlan dense_plan(int64_t M, int64_t m, int64_t k) {
  double us = 0, rest_us = 0;
  const double ring = ring_us(M, m, k);
  const SmallTile* tile = best_small_tile(M, m, k, &us);
  const int64_t nb = m / 256, rounds = ceil_div(ceil_div(M, 128) * nb, 256);
  if (rounds == 1 && k > 8192) us = std::max(us, (double)(m * k) * (17.0 / 32) / 4e6);
  if (tile && us < 0.9 * ring) return {0, tile};
  const int64_t blocks = 256 * (rounds - 1) / nb;  // whole blocks in all rounds but the last
  if (blocks > 0 && (tile = best_small_tile(M - 128 * blocks, m, k, &rest_us)) &&
      ring_us(128 * blocks, m, k) + rest_us < (k >= 4096 ? 0.94 : 0.87) * ring)
    return {128 * blocks, tile};
  return {M, nullptr};
}

// Small tiles of the MXFP8 x MXFP8 GEMM (kern_mx_gemm_mxfp8_t{rows}x{weights}); the fit of their times and of
// kern_mx_gemm_mxfp8's is over 78 shapes (M = 16..1187, N = 512..9216, K = 512..7936; rms 11% and 8%). A tile costs by
// its token subtiles (mt) and 16-row weight groups (n) for every eight k-tiles, one of each wave. A tile is taken where
// the fit has it 15% shorter (its error), in three and more rounds 28% (there its error grows: M = 524, N = 7296,
// K = 960, 1254 tiles of 48 x 64 took 23.0 us against the large tiles' 18.6). Over 8582 shapes (M = 1..6144,
// N = 16..20480, K = 128..16384) the choice takes 0.34 of the large tiles' time, is within 1% of the fastest on average,
// and never slower than the large tiles; with 15% at any number of rounds 16 were, by up to 24%. Over 3353 with N up to
// 160000 or K up to 65536 25 are more than 3% slower, 17% at worst.
struct SmallTile8 {
  int rows, weights;
  const char* entry;
};
#define KERN_SMALL_TILE8(R, W) \
  { R, W, "kern_mx_gemm_mxfp8_t" #R "x" #W }
static const SmallTile8 kSmallTiles8[] = {
    KERN_SMALL_TILE8(16, 16),  KERN_SMALL_TILE8(16, 32), KERN_SMALL_TILE8(16, 64), KERN_SMALL_TILE8(32, 64),
    KERN_SMALL_TILE8(32, 128), KERN_SMALL_TILE8(48, 64), KERN_SMALL_TILE8(64, 64),
};
#undef KERN_SMALL_TILE8
inline const SmallTile8* small_tile8(int64_t m, int64_t n, int64_t k) {
  const int64_t kt = ceil_div(k, 128), big = ceil_div(m, 128) * ceil_div(n, 256);
  const double large =
      5.2 + 0.93 * (double)ceil_div(big, 256) * (double)kt + (double)big / 256 * (8.4 + 0.134 * (double)kt);
  const SmallTile8* best = nullptr;
  double us = 0, most = 0;  // the fastest tile's time, and the longest with which a tile of its rounds is taken
  for (const SmallTile8& t : kSmallTiles8) {
    if (ceil_div(m, t.rows) > 65535 || k > 1 << 20) continue;  // grid.y; 32-bit offsets within a tile
    const double rounds = (double)ceil_div(ceil_div(m, t.rows) * ceil_div(n, t.weights), 256);
    const double mt = t.rows / 16, ng = t.weights / 16;
    const double per8 = -0.046 + 0.304 * mt + 0.176 * ng + 0.0054 * mt * ng;
    const double u = 1.8 + 0.11 * (rounds - 1) + rounds * (0.075 * mt * ng + (double)ceil_div(kt, 8) * per8);
    if (!best || u < us) best = &t, us = u, most = (rounds <= 2 ? 0.85 : 0.72) * large;
  }
  return best && us < most ? best : nullptr;
}

// The decode GEMV at K <= 8192: row groups (kern_mx_gemv_bf16_r{K/512}: one workgroup per 16 weight rows, each reading
// all of x into its LDS) or the persistent walk (p{..}: x read once per workgroup, of which there are about 256). Over
// 1793 shapes (M = 1, 2, 3, 4, 5, 6, 8, 10, 12, 16, eleven N = 1024..18432, every K; graph replays) the choice is within
// 0.5% of the faster on average.
//   M <= 3: row groups at any N (M = 1, N = 2048: 0.71 of the walk's time, N = 18432: 0.94). At M = 3, N > 8192 the
//   walk is ahead at long K (K >= 6144: by 8% on average, 18% at N = 18432, K = 8192; over all K by 2%).
//   M > 3: row groups while they all run at once, N <= 4096 per workgroup of their LDS that a CU holds, at most two
//   (M = 5, N = 3584, K = 7680: 5.4 against 7.7 us), else the walk (M = 8, N = 7168, K = 7680: 9.2 against 10.1 us;
//   M = 16, N = 8192, K = 2560: 5.8 against 8.5; M = 15 there, where one fits: 6.0 against 8.4). At M = 12..16,
//   N = 6144..8192 and K <= 3072 the walk would still be 10% to 21% ahead (M = 12, N = 8192, K = 3072: 5.6 against
//   6.8). At K = 512 it is from N = 4096 on (M = 16, N = 7168: 3.4 against 3.9 us).
// LDS of a row group's workgroup beside x: the waves' sums and (kg + 6) / 4 scale fragments for each wave
inline int64_t gemv_row_group_lds(int64_t kg) { return 4096 + 1024 * ((kg + 6) / 4); }
inline bool gemv_row_groups(int64_t M, int64_t N, int64_t K) {
  const int64_t kg = K / 512, x = 2 * M * K;
  if (kg > 16 || x > 144 * 1024) return false;
  if (M <= 3) return true;
  return N <= 4096 * std::min<int64_t>(2, 163840 / (x + gemv_row_group_lds(kg))) && (kg > 1 || N <= 4096);
}

// Past N = 18432 the walk's workgroups, nine half groups each, need a second round, and the slice-staging kernel
// (kern_mx_gemv_bf16, one workgroup per row group at any N; K > 8192 runs on it anyway) may be ahead: M = 4, N = 19312,
// K = 6144 14.7 against 18.7 us, but M = 16, N = 35904, K = 3584 26.1 against 18.2. Both times fitted to 13285 shapes
// (M = 4..16, N up to 180000, every weight from HBM, the eleven K that took slice staging before the walk had them; rms
// 5%). Over 8291 others of every K and M the choice takes 0.93 of the time of what they took then, at worst 11% more, and
// more than 3% at 58 of them. At K = 512 * {2, 4, 8, 14, 16} the walk stays.
inline int64_t gemv_slice(int64_t M, int64_t kg) {  // k-tiles per wave staged at once: divides kg, M * slice <= 16
  int64_t sb = std::min<int64_t>(kg, 16 / M);
  while (kg % sb) --sb;
  return sb;
}
inline bool gemv_staged(int64_t M, int64_t N, int64_t K) {
  const int64_t kg = K / 512, ktw = (kg + 1) / 2;
  if (kg > 16) return true;
  if (N <= 18432 || kg == 2 || kg == 4 || kg == 8 || kg == 14 || kg == 16) return false;
  const double n = (double)N / 4096, m = (double)M, g = (double)kg, t = (double)ktw;
  const double staged = 4.2 + n * (0.12 + 0.1256 * g + 0.0138 * g * m + 0.0096 * g / (double)gemv_slice(M, kg) - 0.006 * m);
  const double walk =
      2.8 + (double)ceil_div(N, 18432) * (0.5 + 0.69 * t + 0.0176 * t * m) + n * (-0.1 + 0.1 * g + 0.0009 * g * m);
  return staged < 1.03 * walk;
}

}  // namespace kern

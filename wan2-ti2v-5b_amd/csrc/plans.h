// How launches are laid out: sizes in, tiles, parts and grids out.  Host arithmetic only, so that
// it can be checked over any sizes without a device.
#pragma once

#include <cstddef>
#include <cstdint>

namespace wan {

// ---------------------------------------------------------------------------
// the attention (flash_fwd.hip)
// ---------------------------------------------------------------------------

constexpr int kAttnWaves = 8, kTileKeys = 64;   // waves per workgroup (32 query rows each), keys per tile
// A split part's result: per wave (32 query rows) 16 groups of 64 x 4 fp32 (group 4 md + g
// holds o[md][4g..4g+3] of every lane, so that one store writes 1 KB), then m and l per lane.
constexpr int kPartFloats = 64 * 64 + 128;

// How the 8-wave kernel's last round of workgroups (one per CU) is split.  When the blocks
// leave `rem` of them for a last round and that fills half of the CUs at most, each of
// those is run as n workgroups over a part of the keys and merged.  A tile less costs ~1.4 us
// less; a split costs ~5 us (the merge launch, the parts' own start) and 0.05 us per part
// (132 KB of fp32 written and read).  Self-attention, batch 2, 24 heads, us unsplit / split:
//   1500 tokens (rem 32, n 8)  107.6 / 92.6      2048 (rem 128, n 2)  139.4 / 132.8
//   4114 (rem 48, n 5)         482.1 / 437.3
// More than one round of parts loses: 4862 tokens (rem 144) 576 / 581 at n 3, 7854 (rem 208)
// 1382 / 1411 at n 2 -- while a last round is partly idle the busy CUs clock higher.
// The best n is not monotone in the keys (rem 32: 65 tiles in 6 parts, 64 in 8), and the scratch was
// sized for all keys of the tensor where the launch may be given fewer: n is what `scratch` holds.
struct SplitPlan {
  int from, blocks, splits;   // whole blocks, split blocks, parts of each
  size_t bytes;
};
constexpr int kMaxSplits = 8;
inline SplitPlan split_plan(int B, int H, int Lq, int keys, int cus, size_t scratch) {
  SplitPlan p{0, 0, 1, 0};
  const int64_t blocks = (int64_t)((Lq + kAttnWaves * 32 - 1) / (kAttnWaves * 32)) * B * H;
  const int rem = (int)(blocks % cus), nt = (keys + kTileKeys - 1) / kTileKeys;
  if (rem == 0 || blocks > 0x7fffffff) return p;
  const size_t part = (size_t)rem * kAttnWaves * kPartFloats * sizeof(float);   // bytes, one part of each block
  float best = 0.f;
  for (int n = 2; part * n <= scratch && n <= kMaxSplits && rem * n <= cus && n <= nt; ++n) {
    const float gain = 1.4f * (nt - (nt + n - 1) / n) - 5.f - 0.05f * (rem * n);
    if (gain > best) {
      best = gain;
      p.splits = n;
    }
  }
  if (p.splits < 2) return p;
  p.from = (int)(blocks - rem);
  p.blocks = rem;
  p.bytes = part * p.splits;
  return p;
}

// ---------------------------------------------------------------------------
// the token-row kernels (prep.hip, adaln.hip)
// ---------------------------------------------------------------------------

// Their blocks: the W waves of one token row, with a wave a row (W = 1) four rows.
constexpr int rows_per_block(int W) { return W == 1 ? 4 : 1; }
constexpr int row_threads(int W) { return 64 * W * rows_per_block(W); }

// The grid of `blocks` workgroups of `threads`.  A launch has fewer than 2^32 threads along x (22
// million rows of 3072 channels at three waves a row): what is over goes on along y, with up to a
// line's last workgroups too many.
struct RowGrid {
  uint32_t x, y;
};
inline RowGrid row_grid(int64_t blocks, int threads) {
  const int64_t line = 0xffffffffll / threads, y = (blocks + line - 1) / line;
  return {(uint32_t)((blocks + y - 1) / y), (uint32_t)y};
}

// ---------------------------------------------------------------------------
// the projection GEMM (gemm.hip)
// ---------------------------------------------------------------------------

// Columns of an output tile and k per stage.
constexpr int kGemmCols = 256, kGemmBK = 64;

// Tile heights: the x rows of a workgroup's tile, and what a full round of such tiles (one
// workgroup per CU) takes, in us: per 64 of k, and besides (fitted over M 40 to 15708).
constexpr struct { int rows; float k_us; bool power; } kTiles[] = {
    {320, 1.86f, true}, {256, 1.55f, true}, {192, 1.32f, true}, {128, 0.81f, false}};
constexpr float kRoundUs = 6.f;
// A round that fills only a share of the CUs runs at a higher clock (256 rows, N 9216: a second
// round of 0.11, 0.27, 0.55, 0.69 and 0.97 of the CUs takes 54, 58, 62, 67 and 83 us, a full one
// 78); tiles of 128 rows wait for their copies and gain nothing.
inline float round_share(float fill, bool power) { return power ? 0.66f + 0.25f * fill + 0.1f * fill * fill : 1.f; }
// The merge launch, and the write and read of a part's row of 256 fp32 (plain stores: past the
// L2s, non-temporally, the calls took 3-7 us longer).
constexpr float kMergeUs = 4.f, kMergeRowUs = 2 * 256 * 4 / 8e6f;
constexpr int kGemmMaxSplits = 16, kMinSplitTiles = 4;

// The rows of a tile of x are copied from 32-bit byte offsets of its first: whether the last row's
// last byte has one.  wan_qkv_proj_sumsq takes row strides below 2^23 elements, with which it has
// in tiles of up to 256 rows; 320 rows end at 6731920 elements.
inline bool tile_addressable(int M, int rows, int64_t ldx) {
  return (int64_t)((M < rows ? M : rows) - 1) * ldx * 2 + kGemmBK * 2 <= int64_t(1) << 32;
}

// How a product is run: tiles of `rows` rows, the first `from` of them whole, the `rest` as
// `splits` parts over k each.
struct GemmPlan {
  int rows, from, rest, splits;
  float us;
};

// The plan whose rounds take least, with up to `scratch` bytes for the parts, for x rows `ldx`
// elements apart.  Between two heights the number of rounds decides, and where a last (or only)
// round leaves half of the CUs or more idle, its tiles may be split over k: the parts' fp32 sums
// cost a merge launch and their way through memory.  us, tiles of 256 rows alone / as chosen here:
//   N 9216, K 3072:   M 80  56 / 23   M 256  58 / 28   M 896  60 / 46   M 2170  136 / 98 (320 rows)
//                     M 2280  136 / 120 (a tail of 68 tiles, three parts)   M 2940  143 (256 rows)
//                     M 4480  222 / 185 (320)   M 8228  375 / 360 (320)   M 15708  690 / 680
//   N 3072, K 14336 (the best height unsplit / as chosen):   M 80  182 / 36   M 748  178 / 82
//                     M 1500  173 / 132   M 2160  187 / 172 (320 rows, three parts)   M 8228  739 / 581
inline GemmPlan gemm_plan(int M, int N, int K, int64_t ldx, int cus, size_t scratch) {
  GemmPlan best{0, 0, 0, 1, 0.f};
  const int kt = K / kGemmBK;
  for (const auto& t : kTiles) {
    if (!tile_addressable(M, t.rows, ldx)) continue;
    const int64_t tiles = ((int64_t)M + t.rows - 1) / t.rows * (N / kGemmCols);
    const int64_t full = tiles / cus;
    const int rest = (int)(tiles % cus);
    for (int n = 1; n == 1 || (rest > 0 && n <= kGemmMaxSplits && rest * n <= cus && n * kMinSplitTiles <= kt); ++n) {
      if (n > 1 && (size_t)rest * n * t.rows * kGemmCols * sizeof(float) > scratch) break;
      float us = full * (kt * t.k_us + kRoundUs);
      if (rest > 0) us += ((kt + n - 1) / n * t.k_us + kRoundUs) * round_share((float)(rest * n) / cus, t.power);
      if (n > 1) us += kMergeUs + (float)rest * n * t.rows * kMergeRowUs;
      if (best.rows == 0 || us < best.us) best = {t.rows, n > 1 ? (int)(tiles - rest) : 0, n > 1 ? rest : 0, n, us};
    }
  }
  return best;
}

inline size_t gemm_plan_bytes(const GemmPlan& p) {
  return p.splits > 1 ? (size_t)p.rest * p.splits * p.rows * kGemmCols * sizeof(float) : 0;
}

}  // namespace wan

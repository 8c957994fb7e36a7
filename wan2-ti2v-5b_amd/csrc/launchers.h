// Launchers of the kernels around the attention (prep.hip, adaln.hip, gemm.hip): their
// argument blocks and entry points (internal, C++ linkage), called by capi.hip.
#pragma once

#include "common.h"
#include "plans.h"

namespace wan {

// The number of a row kernel's workgroup: its grid goes on along y where x ends (row_grid), `grid_x`
// workgroups to a line.
__device__ __forceinline__ int64_t row_block(unsigned grid_x) { return (int64_t)blockIdx.y * grid_x + blockIdx.x; }

// The sum of v over the W waves that work on one token row; `slot` names a sum of its own
// where a kernel forms several (W = 1: the wave alone, no barrier).
template <int W>
__device__ __forceinline__ float row_sum(float v, int slot) {
  v = wave_sum(v);
  if constexpr (W == 1) {
    return v;
  } else {
    __shared__ float part[2][W];
    if ((threadIdx.x & 63) == 0) part[slot][threadIdx.x >> 6] = v;
    __syncthreads();
    float t = part[slot][0];
#pragma unroll
    for (int i = 1; i < W; ++i) t += part[slot][i];
    return t;
  }
}

struct PrepArgs {
  Tensor4 x;            // input rows [B, L, H, 128]
  int B, L, H;
  float eps;
  float* inv_rms;       // out [B*L] fp32 (may be null)
  const bf16* gamma;    // [H*128] (null: no normalisation applied to `out`)
  const float* cos;     // [L, 64] fp32 (null: no rotation)
  const float* sin;
  bf16* out;            // out [B, L, H, 128] contiguous (null: statistics only)
  // Sums of squares given by the projection GEMM instead of computed from x:
  // partials sumsq[(sumsq_first + p) * B * L + token], p < sumsq_parts (null: from x).
  const float* sumsq;
  int sumsq_first, sumsq_parts;
  unsigned grid_x;      // workgroups along x of the launch (set by the launcher)
};
int launch_rms_prep(const PrepArgs& a, hipStream_t s);
// Two tasks with the same H in one launch.
int launch_rms_prep2(const PrepArgs& a0, const PrepArgs& a1, hipStream_t s);

struct RopeArgs {
  Tensor4 x;
  int B, L, H;
  const float* cos;     // [L, 64]
  const float* sin;
  bf16* out;            // [B, L, H, 128] contiguous
};
int launch_rope(const RopeArgs& a, hipStream_t s);

// One adaLN stage of a block: residual update, LayerNorm, per-frame modulation.
struct AdaLNArgs {
  const bf16* x;        // [B, L, C] residual stream
  const bf16* y;        // [B, L, C] branch output added to x (null: none)
  bf16* x_out;          // [B, L, C] updated residual (null: not written)
  bf16* h_out;          // [B, L, C] normalised (and modulated) row (null: no LayerNorm)
  int B, L, C, F;       // F frames of L / F contiguous tokens each
  const bf16* e;        // [F, 6, C] modulation rows (block modulation + time projection)
  int gate_idx;         // row of e gating y (-1: ungated)
  const bf16* e_mod;    // [F, mod_rows, C] rows of the shift and scale (another block's, or
  int mod_rows;         // the output head's); e with 6 rows when the stage uses its own
  int shift_idx;        // rows of e_mod for the modulation (-1: none)
  int scale_idx;
  const bf16* ln_w;     // [C] LayerNorm affine weight / bias (null: not affine)
  const bf16* ln_b;
  float eps;
  unsigned grid_x;      // workgroups along x of the launch (set by the launcher)
};
int launch_adaln(const AdaLNArgs& a, hipStream_t s);

// out = bf16(x w^T + bias) with per-head sums of squares of the first sq_cols columns.
struct GemmArgs {
  const bf16* x;        // [M, K] (row stride ldx)
  const bf16* w;        // [N, K] (row stride ldw), an nn.Linear weight
  const bf16* bias;     // [N]
  bf16* out;            // [M, N] (row stride ldo)
  float* sumsq;         // [sq_cols / 64, M]: per 64 columns, sum of bf16(out)^2
  int M, N, K;
  int64_t ldx, ldw, ldo;
  int sq_cols;          // multiple of 64, <= N
  // Split of the last round of tiles over k: scratch given by the caller (null: none), and what
  // the launcher makes of it: tiles before split_from are whole, those from there on are
  // `splits` workgroups each that leave their fp32 sums in `part`.
  float* part;
  size_t part_bytes;
  int split_from, splits;
};
// Scratch bytes that a product of this size makes use of (0: it does not split).
size_t gemm_split_bytes(int M, int N, int K);
int launch_gemm_rowsq(const GemmArgs& a, hipStream_t s);

}  // namespace wan

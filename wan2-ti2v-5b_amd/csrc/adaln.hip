// The pointwise chain around a WanAttentionBlock's GEMMs, fused into one pass
// per stage (adaLN: residual update, LayerNorm, per-frame modulation):
//
//   r = x                          (y absent)
//   r = bf16(x + y)                (y, no gate)
//   r = bf16(x + bf16(y * g[f]))   (y, gate row g = e[f, gate_idx])
//   ln = bf16(LayerNorm(r))        fp32 mean / biased variance over the dim channels,
//                                  [* w + b] when the norm is affine
//   h = ln                         (no modulation)
//   h = bf16(bf16(ln * bf16(1 + m[f, scale_idx])) + m[f, shift_idx])
//
// The modulation rows m are e itself, or another row set: the next block's rows when
// one pass ends a block (gated residual) and starts the next (norm1 + modulate), or
// the output head's two rows per frame after the last block.
//
// f is the frame of the token (tokens of one frame are contiguous).  The
// rounding points are those of the reference's eager bf16 graph:
//   _modulate / _gate      models/fast_dit.py:172-181
//   WanLayerNorm           wan/modules/model.py:89-99 (LayerNorm on bf16 input)
//   their use in a block   models/fast_dit.py:280,294,300-311
// so the fused pass equals the separate torch ops except where the order of
// the fp32 LayerNorm sums flips one bf16 rounding.  FMA contraction is off.
//
// Memory bound: a token row is held in registers between the statistics and the
// output; 16-byte loads and stores.
#include "launchers.h"

namespace wan {

namespace {

// W waves work on a token row, each lane on NCH chunks of 8 channels (C <= 512 W NCH).  Two
// chunks a lane and one row a block (three waves at 3072 channels): with a row in one wave, the
// loads in flight of a CU did not cover the latency; with one chunk a lane the barriers of the
// two sums weigh more.  Stages at 3072 channels, us with 1 / 3 / 6 waves a row:
//   gate + modulate   80 rows 8.4 / 4.2 / 3.7   2160 rows 17.8 / 13.8 / 15.3   15708 rows 88 / 77 / 84
//   norm + modulate   80 rows 6.2 / 3.5 / 3.3   2160 rows 11.0 /  8.7 / 10.6   15708 rows 49 / 41 / 55
// STREAM: the tensors of the call exceed what the cache in front of the memory keeps; then x and
// y are read non-temporally and h, which a GEMM reads next, is stored plainly (15708 rows, gate +
// modulate 77 -> 71 us = 5.4 TB/s).  Otherwise both results leave with non-temporal stores: no
// XCD's L2 keeps them for the next kernel, and the launch does not end with their write-back
// (2160 rows, gate + modulate 13.6 -> 12.0 us, norm 8.6 -> 7.4; 8228 rows 41 -> 35).
template <int NCH, int W, bool STREAM>
__global__ __launch_bounds__(row_threads(W)) void adaln_kernel(const AdaLNArgs a) {
  // No contraction into FMAs: each product and sum is rounded to bf16 where the
  // separate torch ops round it (the compiler otherwise fuses ln * s1 + shift
  // across the intermediate bf16 conversion).
#pragma clang fp contract(off)
  const int t = W == 1 ? threadIdx.x & 63 : threadIdx.x;
  const int64_t block = row_block(a.grid_x);
  const int64_t tok = W == 1 ? block * 4 + (threadIdx.x >> 6) : block;
  if (tok >= (int64_t)a.B * a.L) return;
  const int l = (int)(tok % a.L);
  const int f = l / (a.L / a.F);
  const int C = a.C, nch = C >> 3;
  const int64_t row = tok * C;
  const bf16* erow = a.e + (int64_t)f * 6 * C;
  const bf16* mrow = a.e_mod + (int64_t)f * a.mod_rows * C;
  const auto load = [](const bf16* p) {
    const bf16x8* v = reinterpret_cast<const bf16x8*>(p);
    return STREAM ? __builtin_nontemporal_load(v) : *v;
  };

  // every load of the residual update goes out before its first use
  bf16x8 xv[NCH], yv[NCH], gv[NCH];
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int c = t + 64 * W * i;
    if (c < nch) {
      xv[i] = load(a.x + row + 8 * c);
      if (a.y != nullptr) yv[i] = load(a.y + row + 8 * c);
    }
  }
  if (a.y != nullptr && a.gate_idx >= 0) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = t + 64 * W * i;
      if (c < nch) gv[i] = *reinterpret_cast<const bf16x8*>(erow + a.gate_idx * C + 8 * c);
    }
  }

  float r[NCH][8];
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int c = t + 64 * W * i;
    if (c < nch) {
      bf16x8 rv = xv[i];
      if (a.y != nullptr) {
        if (a.gate_idx >= 0) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const bf16 yg = (bf16)((float)yv[i][j] * (float)gv[i][j]);
            rv[j] = (bf16)((float)xv[i][j] + (float)yg);
          }
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) rv[j] = (bf16)((float)xv[i][j] + (float)yv[i][j]);
        }
        if (a.x_out != nullptr) __builtin_nontemporal_store(rv, reinterpret_cast<bf16x8*>(a.x_out + row + 8 * c));
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        r[i][j] = (float)rv[j];
        sum += r[i][j];
      }
    }
  }
  if (a.h_out == nullptr) return;

  const float mean = row_sum<W>(sum, 0) / (float)C;
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    if (t + 64 * W * i < nch) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float d = r[i][j] - mean;
        sq += d * d;
      }
    }
  }
  const float rstd = rsqrtf(row_sum<W>(sq, 1) / (float)C + a.eps);

#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int c = t + 64 * W * i;
    if (c < nch) {
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = rstd * (r[i][j] - mean);
      if (a.ln_w != nullptr) {
        const bf16x8 wv = *reinterpret_cast<const bf16x8*>(a.ln_w + 8 * c);
        const bf16x8 bv = *reinterpret_cast<const bf16x8*>(a.ln_b + 8 * c);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = v[j] * (float)wv[j] + (float)bv[j];
      }
      bf16x8 hv;
      if (a.shift_idx >= 0) {
        const bf16x8 sh = *reinterpret_cast<const bf16x8*>(mrow + a.shift_idx * C + 8 * c);
        const bf16x8 sc = *reinterpret_cast<const bf16x8*>(mrow + a.scale_idx * C + 8 * c);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const bf16 ln = (bf16)v[j];
          const bf16 s1 = (bf16)(1.0f + (float)sc[j]);
          const bf16 u = (bf16)((float)ln * (float)s1);
          hv[j] = (bf16)((float)u + (float)sh[j]);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) hv[j] = (bf16)v[j];
      }
      bf16x8* hp = reinterpret_cast<bf16x8*>(a.h_out + row + 8 * c);
      if (STREAM) *hp = hv;
      else __builtin_nontemporal_store(hv, hp);
    }
  }
}

template <int NCH, int W, bool STREAM>
int launch(AdaLNArgs a, hipStream_t s) {
  const int64_t tokens = (int64_t)a.B * a.L;
  const RowGrid grid = row_grid((tokens + rows_per_block(W) - 1) / rows_per_block(W), row_threads(W));
  if (grid.y > 0xffff) return set_error(2, "adaln: %lld tokens is too many", (long long)tokens);
  a.grid_x = grid.x;
  hipLaunchKernelGGL((adaln_kernel<NCH, W, STREAM>), dim3(grid.x, grid.y), dim3(row_threads(W)), 0, s, a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : set_error(4, "adaln launch: %s", hipGetErrorString(e));
}

// A call whose tensors take more than this is streamed (the last-level cache holds 256 MB).
constexpr int64_t kStreamBytes = int64_t(256) << 20;

template <int NCH, int W>
int launch_w(const AdaLNArgs& a, hipStream_t s) {
  const int tensors = 1 + (a.y != nullptr) + (a.x_out != nullptr) + (a.h_out != nullptr);
  return (int64_t)a.B * a.L * a.C * 2 * tensors > kStreamBytes ? launch<NCH, W, true>(a, s)
                                                               : launch<NCH, W, false>(a, s);
}

}  // namespace

int launch_adaln(const AdaLNArgs& a, hipStream_t s) {
  if ((int64_t)a.B * a.L == 0) return 0;
  if (a.C <= 512) return launch_w<1, 1>(a, s);
  if (a.C <= 1024) return launch_w<2, 1>(a, s);
  if (a.C <= 2048) return launch_w<2, 2>(a, s);
  if (a.C <= 3072) return launch_w<2, 3>(a, s);
  if (a.C <= 4096) return launch_w<2, 4>(a, s);
  return launch_w<2, 8>(a, s);
}

}  // namespace wan

// Token-row kernels of the attention path: the QK-RMSNorm statistics (and the
// normalised, rotated K rows the attention kernel streams), and a standalone
// 3D-RoPE rotation.
//
// Rounding follows the reference's bf16 graph exactly:
//   _tp_rms_qk  models/fast_dit.py:134-147   t = bf16(x * rsqrt(sum(x^2)/C + eps)); u = bf16(t * gamma)
//   _rope       models/fast_dit.py:163-169   fp32 pair rotation of u, one bf16 rounding
// Contraction into FMAs is disabled in the rotation so each product and sum is
// rounded as the separate torch ops round it.
#include "launchers.h"

#include <algorithm>

namespace wan {

namespace {

constexpr int kMaxChunksPerLane = 16;  // supports H*128 <= 8192 channels per token

// A task that only turns given partial sums into inverse RMS.
__host__ __device__ inline bool sums_only(const PrepArgs& a) { return a.sumsq != nullptr && a.out == nullptr; }

// Rotate interleaved pairs of 8 consecutive channels of one token by their four angles.
__device__ __forceinline__ void rope8(float u[8], const f32x4 c, const f32x4 s) {
#pragma clang fp contract(off)
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float xr = u[2 * j], xi = u[2 * j + 1];
    const float a = xr * c[j];
    const float b = xi * s[j];
    const float e = xr * s[j];
    const float f = xi * c[j];
    u[2 * j] = a - b;
    u[2 * j + 1] = e + f;
  }
}

// Sum of squares over all H*128 channels of a token row, then optionally the normalised (and
// rotated) row.  W waves work on a row, each lane on NCH chunks of 8 channels (H*16 <= 64 W NCH).
// With W > 1 a block is one row, with W = 1 (up to 1024 channels) four.  A row in one wave was
// latency bound: too few loads in flight a CU, and for few rows one wave's chain of loads, 48
// channels of arithmetic a lane and stores was what the launch took.  At 3072 channels, us with
// 1 / 3 / 6 waves a row (the kernels of a call as the launcher chooses now):
//   norm + rotation   748 rows 6.1 / 5.2 / 4.7   2160 rows 10.3 / 8.4 / 8.8   15708 rows 41.9 / 36.6 / 47.1
//   statistics        748 rows 4.1 / 3.4 / 3.4   2160 rows  5.4 / 5.0 / 5.9   15708 rows 20.2 / 17.6 / 26.7
// All loads go out before the sum is formed.
// NT: non-temporal stores of the normalised rows.  No XCD's L2 keeps them for the next kernel,
// and the launch does not end with their write-back (norm + rotation 2160 rows 8.4 -> 7.0 us,
// 8228 rows 22.0 -> 20.1); with more than the last-level cache takes of rows read and written
// they cost (15708 rows 36.6 -> 38.9).
// NTR: non-temporal reads of the rows, in the launches of both tasks that write too much to keep (q,
// k and the written k are 289 MB at 15708 rows, the last-level cache is 256 MB).  Plain reads take
// lines there that others have written, which must go to memory first, and put out what the next
// kernel would have found.  15708 rows, us plain / so: the pass behind 512 MB of other writes 93 / 54, behind
// a GEMM of other rows 61 / 53, the projection GEMM (256 rows, unsplit) behind the pass 749 / 684; behind the
// rows' own projection, with the attention after it, 1337 / 1338.  Smaller launches, and the statistics
// alone, read plainly: the attention finds q in the cache (2 x 1080 tokens, pass and attention
// 53.1 / 54.0 us; statistics and cross-attention of 15708 rows 135.9 / 138.1).
template <int NCH, int W, bool NT, bool NTR>
__device__ __forceinline__ void rms_prep_rows(const PrepArgs& a, unsigned block) {
  const int t = W == 1 ? threadIdx.x & 63 : threadIdx.x;
  const unsigned row_id = W == 1 ? block * 4 + (threadIdx.x >> 6) : block;
  if (row_id >= (unsigned)(a.B * a.L)) return;
  const int tok = (int)row_id;
  const int b = tok / a.L, l = tok - b * a.L;
  const int nchunks = a.H * 16;
  const bf16* row = a.x.ptr + b * a.x.sb + (int64_t)l * a.x.st;
  const bool want = a.out != nullptr;

  bf16x8 xv[NCH], gv[NCH];
  float ss = 0.f;
  // with the projection GEMM's partial sums the row is read only when it is to be normalised
  if (want || a.sumsq == nullptr) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = t + 64 * W * i;
      if (c < nchunks) {
        const bf16x8* xp = reinterpret_cast<const bf16x8*>(row + (c >> 4) * a.x.sh + (c & 15) * 8);
        xv[i] = NTR ? __builtin_nontemporal_load(xp) : *xp;
      }
    }
  }
  // the channel pairs of a lane's chunks are the same in every head: 64 W is a multiple of 16
  const int d0 = (t & 15) * 8;
  f32x4 cs = {}, sn = {};
  if (want) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = t + 64 * W * i;
      if (c < nchunks) gv[i] = *reinterpret_cast<const bf16x8*>(a.gamma + 8 * c);
    }
    if (a.cos != nullptr) {
      cs = *reinterpret_cast<const f32x4*>(a.cos + (int64_t)l * kRopePairs + d0 / 2);
      sn = *reinterpret_cast<const f32x4*>(a.sin + (int64_t)l * kRopePairs + d0 / 2);
    }
  }
  if (a.sumsq != nullptr) {
    // one partial sum a lane (64 at most) of the row's first wave
    if (t < a.sumsq_parts) ss = a.sumsq[(int64_t)(a.sumsq_first + t) * (a.B * a.L) + tok];
  } else {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      if (t + 64 * W * i < nchunks) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float f = (float)xv[i][j];
          ss += f * f;
        }
      }
    }
  }
  ss = row_sum<W>(ss, 0);
  const float inv = 1.0f / sqrtf(ss / (float)(a.H * kHeadDim) + a.eps);
  if (a.inv_rms != nullptr && t == 0) a.inv_rms[tok] = inv;
  if (!want) return;

  bf16* orow = a.out + (int64_t)tok * a.H * kHeadDim;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int c = t + 64 * W * i;
    if (c < nchunks) {
      float u[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const bf16 n = (bf16)((float)xv[i][j] * inv);
        u[j] = (float)(bf16)((float)n * (float)gv[i][j]);
      }
      if (a.cos != nullptr) rope8(u, cs, sn);
      bf16x8 r;
#pragma unroll
      for (int j = 0; j < 8; ++j) r[j] = (bf16)u[j];
      bf16x8* op = reinterpret_cast<bf16x8*>(orow + 8 * c);
      if (NT) __builtin_nontemporal_store(r, op);
      else *op = r;
    }
  }
}

// The statistics alone, from the projection GEMM's partial sums: a thread per token, so that the
// 64 tokens of a wave read whole lines (us with their k pass, a block per token / so: 2160 tokens
// 8.0 / 7.0, 8228 28.0 / 22.8, 15708 52.3 / 37.7; with a loop of single loads 9.2 / 28.2 / 38.9).
template <int W>
__device__ __forceinline__ void inv_rms_of_sums(const PrepArgs& a, unsigned block) {
  const unsigned tok = block * row_threads(W) + threadIdx.x;
  if (tok >= (unsigned)(a.B * a.L)) return;
  const float* p = a.sumsq + (int64_t)a.sumsq_first * (a.B * a.L) + tok;
  // sixteen sums side by side, then their tree: no partial sum takes part in more than 8 roundings (a
  // wave's tree 6; one chain of 64, 63)
  float t[16] = {};
  int i = 0;
  for (; i + 16 <= a.sumsq_parts; i += 16)
#pragma unroll
    for (int j = 0; j < 16; ++j) t[j] += p[(int64_t)(i + j) * (a.B * a.L)];
#pragma unroll
  for (int j = 0; j < 16; ++j)
    if (i + j < a.sumsq_parts) t[j] += p[(int64_t)(i + j) * (a.B * a.L)];
#pragma unroll
  for (int n = 8; n > 0; n /= 2)
#pragma unroll
    for (int j = 0; j < n; ++j) t[j] += t[j + n];
  const float ss = t[0];
  a.inv_rms[tok] = 1.0f / sqrtf(ss / (float)(a.H * kHeadDim) + a.eps);
}

template <int NCH, int W, bool NT>
__global__ __launch_bounds__(row_threads(W)) void rms_prep_kernel(const PrepArgs a) {
  rms_prep_rows<NCH, W, NT, false>(a, (unsigned)row_block(a.grid_x));
}

// Two independent tasks (the q statistics and the k norm + rotation of one
// self-attention call) in one launch: blocks [0, blocks0) run a0, the rest a1.
template <int NCH, int W, bool NT>
__global__ __launch_bounds__(row_threads(W)) void rms_prep2_kernel(const PrepArgs a0, const PrepArgs a1,
                                                                   unsigned blocks0) {
  const unsigned block = (unsigned)row_block(a0.grid_x);   // (rows, and so blocks, are below 2^31 a task)
  if (block < blocks0) {
    if (sums_only(a0)) inv_rms_of_sums<W>(a0, block);
    else rms_prep_rows<NCH, W, NT, !NT>(a0, block);
  } else {
    rms_prep_rows<NCH, W, NT, !NT>(a1, block - blocks0);
  }
}

// One thread per 8 channels: out = rope(x), the _rope semantics on its own.
__global__ __launch_bounds__(256) void rope_kernel(const RopeArgs a) {
  const int64_t chunk = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t total = (int64_t)a.B * a.L * a.H * 16;
  if (chunk >= total) return;
  const int d0 = (int)(chunk & 15) * 8;
  int64_t rest = chunk >> 4;
  const int h = (int)(rest % a.H);
  rest /= a.H;
  const int l = (int)(rest % a.L);
  const int b = (int)(rest / a.L);
  const bf16x8 x = *reinterpret_cast<const bf16x8*>(a.x.ptr + b * a.x.sb + (int64_t)l * a.x.st +
                                                    h * a.x.sh + d0);
  float u[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) u[j] = (float)x[j];
  rope8(u, *reinterpret_cast<const f32x4*>(a.cos + (int64_t)l * kRopePairs + d0 / 2),
        *reinterpret_cast<const f32x4*>(a.sin + (int64_t)l * kRopePairs + d0 / 2));
  bf16x8 r;
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = (bf16)u[j];
  *reinterpret_cast<bf16x8*>(a.out + chunk * 8) = r;
}

// Up to this many rows in a launch a lane has one chunk of 8 channels, beyond it two.
constexpr int kFewRows = 1024;
// Normalised rows leave with plain stores when rows read and written exceed this many bytes, and the
// launches of both tasks then read non-temporally.
constexpr int64_t kStreamBytes = int64_t(128) << 20;

// Launches `a0` alone (a1 null) or both tasks.
template <int NCH, int W, bool NT>
int launch_prep(PrepArgs a0, const PrepArgs* a1, hipStream_t s) {
  constexpr int R = rows_per_block(W);
  const int per0 = a1 != nullptr && sums_only(a0) ? row_threads(W) : R;
  const int64_t blocks0 = ((int64_t)a0.B * a0.L + per0 - 1) / per0;
  const int64_t blocks1 = a1 != nullptr ? ((int64_t)a1->B * a1->L + R - 1) / R : 0;
  const RowGrid g = row_grid(blocks0 + blocks1, row_threads(W));
  const dim3 grid(g.x, g.y), block(row_threads(W));
  a0.grid_x = g.x;
  if (a1 == nullptr)
    hipLaunchKernelGGL((rms_prep_kernel<NCH, W, NT>), grid, block, 0, s, a0);
  else
    hipLaunchKernelGGL((rms_prep2_kernel<NCH, W, NT>), grid, block, 0, s, a0, *a1, (unsigned)blocks0);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : set_error(4, "rms_prep launch: %s", hipGetErrorString(e));
}

// N: chunks a lane when a row is one wave's.
template <int N>
int launch_prep_n(const PrepArgs& a0, const PrepArgs* a1, hipStream_t s) {
  const int64_t rows = (int64_t)a0.B * a0.L + (a1 != nullptr ? (int64_t)a1->B * a1->L : 0);
  const PrepArgs& last = a1 != nullptr ? *a1 : a0;   // the task that may write rows
  if (rows <= kFewRows) return launch_prep<1, N, true>(a0, a1, s);
  if constexpr (N == 1) return launch_prep<1, 1, true>(a0, a1, s);
  else if ((int64_t)last.B * last.L * last.H * (kHeadDim * 4) > kStreamBytes)
    return launch_prep<2, N / 2, false>(a0, a1, s);
  else return launch_prep<2, N / 2, true>(a0, a1, s);
}

int launch_prep_any(const PrepArgs& a0, const PrepArgs* a1, hipStream_t s) {
  const int nch = a0.H * 16;
  if (nch > 64 * kMaxChunksPerLane) return set_error(2, "rms_prep: H*128=%d channels exceeds 8192", a0.H * 128);
  const int64_t most = std::max((int64_t)a0.B * a0.L, a1 != nullptr ? (int64_t)a1->B * a1->L : 0);
  if (most > 0x7fffffff) return set_error(2, "rms_prep: %lld rows is too many", (long long)most);
  if (nch <= 64) return launch_prep_n<1>(a0, a1, s);
  if (nch <= 128) return launch_prep_n<2>(a0, a1, s);
  if (nch <= 256) return launch_prep_n<4>(a0, a1, s);
  if (nch <= 384) return launch_prep_n<6>(a0, a1, s);
  if (nch <= 512) return launch_prep_n<8>(a0, a1, s);
  return launch_prep_n<16>(a0, a1, s);
}

}  // namespace

int launch_rms_prep(const PrepArgs& a, hipStream_t s) {
  if ((int64_t)a.B * a.L == 0) return 0;
  return launch_prep_any(a, nullptr, s);
}

int launch_rms_prep2(const PrepArgs& a0, const PrepArgs& a1, hipStream_t s) {
  if (a0.H != a1.H) return set_error(1, "rms_prep: the paired tasks differ in heads");
  if ((int64_t)a0.B * a0.L == 0) return launch_rms_prep(a1, s);
  if ((int64_t)a1.B * a1.L == 0) return launch_rms_prep(a0, s);
  return launch_prep_any(a0, &a1, s);
}

int launch_rope(const RopeArgs& a, hipStream_t s) {
  const int64_t total = (int64_t)a.B * a.L * a.H * 16;
  if (total == 0) return 0;
  hipLaunchKernelGGL(rope_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : set_error(4, "rope launch: %s", hipGetErrorString(e));
}

}  // namespace wan

// The block's q/k/v projection as one bf16 GEMM on gfx950, with the statistics of the
// QK-RMSNorm in its epilogue:
//
//   out[m, n]    = bf16(sum_k x[m, k] w[n, k] + bias[n])          (F.linear, models/fast_dit.py:281)
//   sumsq[p, m]  = sum over columns 64 p .. 64 p + 63 of bf16(out[m, n])^2,  for 64 p < sq_cols
//
// so that the per-token sums of squares of q and k over all heads (_tp_rms_qk,
// models/fast_dit.py:134-147) are 48 + 48 partial sums read by the K pass, and q is
// not read again before the attention kernel.
//
// Design: GBM x 256 output tile per workgroup (GBM 128, 192, 256 or 320: the launcher
// takes the height that fills the rounds of workgroups best), 8 waves in a 2 x 4 grid,
// each wave GBM/2 (m) x 64 (n): up to 10 accumulators of v_mfma_f32_32x32x16_bf16, two
// waves per SIMD.  The MFMA computes out^T tiles, w rows on the MFMA row axis and x rows
// on the column axis, so a lane holds one output row (lane % 32) and half of each
// 64-column block: a 64-column sum of squares is lane-local plus one exchange with the
// lane 32 apart, as the attention kernel's softmax row sums are.  K advances 64 per
// tile; the GBM x 64 and 256 x 64 tiles of x and w (32 KB for 256 rows) go global -> LDS
// by 16-byte copies into rows of eight 16-byte chunks, chunk c of row r at position c ^
// ((r / 2) % 8) (conflict-free operand reads), in two slots (three with 128 rows, whose
// 1024 MFMA cycles per tile are less than a copy takes: 46 -> 33 us at M 256), one
// barrier per tile.  (256 rows in 32-k stages, three to five slots: 4-8% slower than 64
// k in two.) Program order is pinned MFMA by MFMA: each MFMA is followed by one fragment
// read of the next k-step and, in a tile's first k-step, one copy of a coming tile, and
// the barrier sits inside the last k-step so the next tile's first reads overlap its
// remaining MFMAs.  Workgroups run in groups of 8 M-tiles per N-tile, each XCD owning a
// contiguous range, so the tiles running together on an XCD share x and w rows in its
// L2.
//
// At the QKV shape (M 15708, N 9216, K 3072) it takes 0.67-0.69 ms as the operators run it (320 rows,
// the tail split over k), 1.29-1.33 PFLOP/s and 88-90% of hipBLASLt's F.linear timed beside it; without
// scratch (256 rows) 0.68-0.70 ms.  At M 2160 (320 rows) 1.29 PFLOP/s against hipBLASLt's 1.17.  Both
// are power
// limited (all-zero operands run either ~25% faster); on zeros this kernel's k-loop is
// ~13% slower per tile than hipBLASLt's.  4 waves of 128 x 128 (a third less LDS read
// traffic, one wave per SIMD) run the loop at a higher clock (1.72 vs 1.58 GHz) but in
// more cycles per tile, and tie with this tiling at best.
#include "launchers.h"
#include "plans.h"

#include <type_traits>

namespace wan {

namespace {

constexpr int GBN = kGemmCols;
constexpr int kGroupM = 8;
// 8 waves in a 2 x 4 grid (each 128 x 64 of a 256 x 256 tile, two waves per SIMD),
// 64 k per stage: measured the fastest of 2 x 2 / 2 x 4 waves, 32 / 64 k, 2-5 stages
constexpr int kGemmWM = 2, kGemmWN = 4;

__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t lds_addr(const bf16* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) bf16*)p;
}

// 16-byte global -> LDS copy (lane l writes LDS bytes m0 + 16 l ..), from inline asm so
// the compiler's LDS wait counting does not see it (see flash_fwd.hip); completion is
// waited for explicitly before the barrier that publishes a stage.  A memory instruction
// needs 5 wait states after a VALU write (v_readfirstlane / v_readlane) of an SGPR it
// reads, and the compiler does not pad that for inline asm: the scalar base of this copy
// and of flash_fwd.hip's must come from scalar code (tests/test_isa_hazards.py checks
// the compiled kernels).
__device__ __forceinline__ void dma16(const char* sbase, uint32_t voff, uint32_t lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(voff), "s"(sbase), "{m0}"(lds) : "memory");
}

__device__ __forceinline__ float pair_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <int WM, int WN, int BK, int GBM>
struct GemmCfg {
  static constexpr int kWaves = WM * WN;
  static constexpr int kThreads = 64 * kWaves;
  static constexpr int TM = GBM / WM / 32;        // 32-row blocks of x (output rows) per wave
  static constexpr int TN = GBN / WN / 32;        // 32-row blocks of w (output columns) per wave
  static constexpr int kCpr = BK / 8;             // 16-byte chunks per tile row
  static constexpr int kRps = 16 / kCpr;          // rows per 256-byte bank sweep
  static constexpr int kRowsPerBlock = 512 / BK;  // tile rows per 1 KB copy
  static constexpr int kXPerWave = GBM / kRowsPerBlock / kWaves;  // 1 KB copies per wave and tile
  static constexpr int kWPerWave = GBN / kRowsPerBlock / kWaves;
  static_assert(GBM % (32 * WM) == 0 && GBN % (64 * WN) == 0, "whole 32-row and 64-column blocks");
  static_assert(GBM % (kRowsPerBlock * kWaves) == 0 && GBN % (kRowsPerBlock * kWaves) == 0,
                "copies must divide over the waves");
  static_assert(2 * GBM * BK >= kWaves * 32 * GBN / WN, "the x tiles hold the output staging");
  // chunk c of row r sits at position c ^ ((r / kRps) % kCpr): the 16 rows read by a
  // 16-lane phase of an operand read land on 16 distinct 16-byte bank groups
  __device__ static __forceinline__ int swz(int row) { return (row / kRps) & (kCpr - 1); }
};

// Copies of one tile of 8 N x BK rows in 1 KB blocks, N per wave, wave w issuing blocks w, w + waves, ...
// Lane l fills LDS row (block rows) + l / kCpr, position l % kCpr, with the global chunk
// the row's swizzle puts there.  Offsets are bytes from the tile's (row 0, k 0).
template <class C, int N>
struct GemmTileLoader {
  uint32_t off[N];
  __device__ void init(int64_t ld, int rows_valid, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int row = C::kRowsPerBlock * (wave + C::kWaves * i) + lane / C::kCpr;
      const int r = min(row, rows_valid - 1);       // rows past the matrix repeat its last row
      off[i] = (uint32_t)((int64_t)r * ld * 2 + (((lane % C::kCpr) ^ C::swz(row)) << 4));
    }
  }
  __device__ __forceinline__ void issue_one(const char* tile_base, bf16* dst, int wave, int i) const {
    dma16(tile_base, off[i], lds_addr(dst + (wave + C::kWaves * i) * 512));
  }
};

// First row and column of output tile `pid`: groups of kGroupM M-tiles, N-tiles within a group.
__device__ __forceinline__ void tile_origin(const GemmArgs& a, int pid, int rows, int& m0, int& n0) {
  const int mt_count = (a.M + rows - 1) / rows, nt_count = a.N / GBN;
  const int per_group = kGroupM * nt_count;
  const int group = pid / per_group, first_m = group * kGroupM;
  const int gsize = min(mt_count - first_m, kGroupM);
  const int in_group = pid - group * per_group;
  m0 = (first_m + in_group % gsize) * rows;
  n0 = in_group / gsize * GBN;
}

// A 32-row block of a wave's columns (64 TN / 2, from column ncol0): the sums of squares over
// each 64 of them and the rounded rows, staged through this wave's LDS (row-major, chunk c of
// row r at position c ^ (r % chunks)) and stored as whole row segments.  `value` gives the
// lane's four values of row l32 from column 32 nb + 8 g + 4 hh of the block on.
template <int TN, typename F>
__device__ __forceinline__ void store_rows32(const GemmArgs& a, int row0, int ncol0, bf16* stage, int lane, F value) {
  constexpr int kCols = TN * 32, kChunks = kCols / 8;
  const int l32 = lane & 31, hh = lane >> 5;
  float ss[TN / 2] = {};
#pragma unroll
  for (int nb = 0; nb < TN; ++nb) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const bf16x4 v = value(nb, g);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float f = (float)v[e];
        ss[nb / 2] = fmaf(f, f, ss[nb / 2]);
      }
      const int c = 4 * nb + g;   // this lane's columns 8c + 4hh .. +3 of row l32
      *reinterpret_cast<bf16x4*>(stage + l32 * kCols + ((c ^ (l32 % kChunks)) << 3) + 4 * hh) = v;
    }
  }
#pragma unroll
  for (int h = 0; h < TN / 2; ++h) {
    const float t = pair_sum(ss[h]);
    if (ncol0 + 64 * h < a.sq_cols && hh == 0 && row0 + l32 < a.M)
      a.sumsq[(int64_t)(ncol0 / 64 + h) * a.M + row0 + l32] = t;
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  constexpr int kRowsPerStore = 64 / kChunks;
#pragma unroll
  for (int j = 0; j < 32 / kRowsPerStore; ++j) {
    const int r = kRowsPerStore * j + lane / kChunks, c = lane % kChunks;
    const bf16x8 v = *reinterpret_cast<const bf16x8*>(stage + r * kCols + ((c ^ (r % kChunks)) << 3));
    if (row0 + r < a.M)
      __builtin_nontemporal_store(v, reinterpret_cast<bf16x8*>(a.out + (int64_t)(row0 + r) * a.ldo + ncol0 + 8 * c));
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

template <int WM, int WN, int BK, int GBM, int SLOTS, bool SPLIT>
__global__ __launch_bounds__(64 * WM * WN, 1) void gemm_rowsq_kernel(const GemmArgs a) {
  using C = GemmCfg<WM, WN, BK, GBM>;
  __shared__ __attribute__((aligned(1024))) bf16 xs[SLOTS][GBM * BK];
  __shared__ __attribute__((aligned(1024))) bf16 ws[SLOTS][GBN * BK];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const int l32 = lane & 31, hh = lane >> 5;

  // Each XCD owns a contiguous range of the tiles, and of the split parts: those part by part,
  // so that the tiles of one k range that run together on an XCD share x and w rows.
  int pid, part = -1, kt_first = 0, kt_count = a.K / BK;
  if (!SPLIT || (int)blockIdx.x < a.split_from) {
    pid = xcd_remap(blockIdx.x, SPLIT ? a.split_from : gridDim.x);
  } else {
    const int n = gridDim.x - a.split_from, tiles = n / a.splits;
    const int i = xcd_remap(blockIdx.x - a.split_from, n);
    const int k = i / tiles, tile = i - k * tiles;
    pid = a.split_from + tile;
    part = tile * a.splits + k;
    kt_first = (int)((int64_t)kt_count * k / a.splits);
    kt_count = (int)((int64_t)kt_count * (k + 1) / a.splits) - kt_first;
  }
  int m0, n0;
  tile_origin(a, pid, GBM, m0, n0);

  GemmTileLoader<C, C::kXPerWave> xl;
  GemmTileLoader<C, C::kWPerWave> wl;
  xl.init(a.ldx, a.M - m0, wave, lane);
  wl.init(a.ldw, GBN, wave, lane);
  const char* xbase = reinterpret_cast<const char*>(a.x + (int64_t)m0 * a.ldx + kt_first * BK);
  const char* wbase = reinterpret_cast<const char*>(a.w + (int64_t)n0 * a.ldw + kt_first * BK);

  // operand rows of this lane within the tiles; (row / kRps) % kCpr is the same for
  // every 32-row block
  int xrow[C::TM], wrow[C::TN];
#pragma unroll
  for (int b = 0; b < C::TM; ++b) xrow[b] = (wm * C::TM + b) * 32 + l32;
#pragma unroll
  for (int b = 0; b < C::TN; ++b) wrow[b] = (wn * C::TN + b) * 32 + l32;
  const int sw = C::swz(l32);

  // the bias of this wave's columns, loaded before the k-loop: in the epilogue its
  // loads stood first on the critical path (1-1.3% of the launch)
  constexpr int kCols = C::TN * 32;              // this wave's columns (64 or 128)
  constexpr bool kEarlyBias = C::TM < 5;         // (with five row blocks there is no register left)
  bf16x4 bias_r[C::TN][4];
  auto load_bias = [&] {
#pragma unroll
    for (int nb = 0; nb < C::TN; ++nb)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        bias_r[nb][g] = *reinterpret_cast<const bf16x4*>(a.bias + n0 + wn * kCols + nb * 32 + 8 * g + 4 * hh);
  };
  if constexpr (kEarlyBias) load_bias();

  f32x16 acc[C::TN][C::TM];
#pragma unroll
  for (int i = 0; i < C::TN; ++i)
#pragma unroll
    for (int j = 0; j < C::TM; ++j) acc[i][j] = f32x16{};

  auto read_frag = [&](int slot, int ks, int i, bf16x8 wf[C::TN], bf16x8 xf[C::TM]) {
    const int pos = ((2 * ks + hh) ^ sw) << 3;
    if (i < C::TN)
      wf[i] = *reinterpret_cast<const bf16x8*>(ws[slot] + wrow[i] * BK + pos);
    else
      xf[i - C::TN] = *reinterpret_cast<const bf16x8*>(xs[slot] + xrow[i - C::TN] * BK + pos);
  };
  auto copy_one = [&](int slot, int kt, int i) {
    const int64_t kb = (int64_t)kt * BK * 2;
    if (i < C::kXPerWave)
      xl.issue_one(xbase + kb, xs[slot], wave, i);
    else
      wl.issue_one(wbase + kb, ws[slot], wave, i - C::kXPerWave);
  };
  constexpr int KS = BK / 16;             // MFMA k-steps per tile
  constexpr int NF = C::TN + C::TM;       // fragment reads per k-step
  constexpr int NM = C::TN * C::TM;       // MFMAs per k-step
  constexpr int NC = C::kXPerWave + C::kWPerWave;  // copies per tile and wave
  constexpr int PRE = NM - NF;            // MFMAs of the last k-step before the barrier
  static_assert(KS % 2 == 0 && NF <= NM, "schedule");

  bf16x8 wf[2][C::TN], xf[2][C::TM];

  // One tile of k.  Program order is fixed MFMA by MFMA (a scheduling barrier after
  // each): after MFMA m of k-step ks comes fragment read m of k-step ks + 1 (the reads
  // are in flight behind the MFMAs that follow) and, in k-step 0, copy m of the tile
  // SLOTS - 1 ahead into the slot that the tile before this one left.  The last k-step
  // splits around the barrier that publishes the next tile: NM - NF MFMAs, the wait for
  // that tile's copies (those of later tiles stay in flight) and the barrier, then NF
  // MFMAs, each followed by a read of the next tile's first k-step.
  int ring = 0;                       // slot of tile kt, with more than two
  auto tile = [&](int kt, auto next_c, auto copy_c) {
    constexpr bool has_next = decltype(next_c)::value, has_copy = decltype(copy_c)::value;
    const int slot = SLOTS == 2 ? kt & 1 : ring;
    const int nslot = SLOTS == 2 ? slot ^ 1 : slot == SLOTS - 1 ? 0 : slot + 1;
    const int cslot = SLOTS == 2 ? slot ^ 1 : slot == 0 ? SLOTS - 1 : slot - 1;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int cur = ks & 1, nxt = cur ^ 1;
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        if (ks == KS - 1 && m == PRE) {
          // every wave's copies of the next tile landed, every read of this slot returned
          if constexpr (has_copy && SLOTS > 2)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "i"((SLOTS - 2) * NC) : "memory");
          else
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
          __builtin_amdgcn_sched_barrier(0);
        }
        const int nb = m / C::TM, mb = m % C::TM;
        acc[nb][mb] = mfma32(wf[cur][nb], xf[cur][mb], acc[nb][mb]);
        if (ks < KS - 1) {
          if (m < NF) read_frag(slot, ks + 1, m, wf[nxt], xf[nxt]);
        } else if (has_next && m >= PRE) {
          read_frag(nslot, 0, m - PRE, wf[nxt], xf[nxt]);
        }
        if (has_copy && ks == 0 && m < NC) copy_one(cslot, kt + SLOTS - 1, m);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (has_copy && ks == 0) {
#pragma unroll
        for (int i = NM; i < NC; ++i) copy_one(cslot, kt + SLOTS - 1, i);
      }
    }
    ring = nslot;
  };

  for (int t = 0; t < SLOTS - 1 && t < kt_count; ++t)
    for (int i = 0; i < NC; ++i) copy_one(t, t, i);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NF; ++i) read_frag(0, 0, i, wf[0], xf[0]);
  using yes = std::integral_constant<bool, true>;
  using no = std::integral_constant<bool, false>;
  int kt = 0;
  for (; kt + SLOTS - 1 < kt_count; ++kt) tile(kt, yes{}, yes{});
  if constexpr (SLOTS > 2)
    for (; kt + 1 < kt_count; ++kt) tile(kt, yes{}, no{});
  tile(kt, no{}, no{});
  if (SPLIT && part >= 0) {
    // fp32, 64 lanes x 4 values a store: block (wave, mb, nb, g) of 1 KB
    float* p = a.part + (int64_t)part * (GBM * GBN) + wave * (C::TM * C::TN * 1024) + lane * 4;
#pragma unroll
    for (int mb = 0; mb < C::TM; ++mb)
#pragma unroll
      for (int nb = 0; nb < C::TN; ++nb)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          f32x4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[nb][mb][4 * g + e];
          *reinterpret_cast<f32x4*>(p + ((mb * C::TN + nb) * 4 + g) * 256) = v;
        }
    return;
  }
  if constexpr (!kEarlyBias) load_bias();
  __syncthreads();   // every wave is done with the last stage before the output staging

  bf16* stage = &xs[0][0] + wave * 32 * kCols;
#pragma unroll
  for (int mb = 0; mb < C::TM; ++mb)
    store_rows32<C::TN>(a, m0 + (wm * C::TM + mb) * 32, n0 + wn * kCols, stage, lane, [&](int nb, int g) {
      bf16x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (bf16)(acc[nb][mb][4 * g + e] + (float)bias_r[nb][g][e]);
      return v;
    });
}

// The output of the split tiles: their parts summed in order, then the epilogue.  One wave per
// 32 rows x 64 columns (a wave's 32-row block of the GEMM), four waves a workgroup.
__global__ __launch_bounds__(256) void gemm_merge_kernel(const GemmArgs a, int rows) {
  constexpr int TN = GBN / kGemmWN / 32;
  __shared__ __attribute__((aligned(16))) bf16 stage[4][32 * TN * 32];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int hh = lane >> 5;
  const int tm = rows / (32 * kGemmWM), per_tile = kGemmWM * kGemmWN * tm;
  const int piece = blockIdx.x * 4 + wave;
  const int tile = piece / per_tile, block = piece - tile * per_tile;
  const int gw = block / tm, mb = block - gw * tm;      // the GEMM's wave and its 32-row block
  int m0, n0;
  tile_origin(a, a.split_from + tile, rows, m0, n0);
  const int row0 = m0 + (gw % kGemmWM * tm + mb) * 32, ncol0 = n0 + gw / kGemmWM * (TN * 32);
  if (row0 >= a.M) return;

  const float* p = a.part + (int64_t)tile * a.splits * (rows * GBN) + block * (TN * 1024) + lane * 4;
  f32x4 acc[TN][4];
#pragma unroll
  for (int i = 0; i < 4 * TN; ++i) acc[i / 4][i % 4] = *reinterpret_cast<const f32x4*>(p + i * 256);
  for (int k = 1; k < a.splits; ++k) {
    p += rows * GBN;
#pragma unroll
    for (int i = 0; i < 4 * TN; ++i) acc[i / 4][i % 4] += *reinterpret_cast<const f32x4*>(p + i * 256);
  }
  store_rows32<TN>(a, row0, ncol0, stage[wave], lane, [&](int nb, int g) {
    const bf16x4 b = *reinterpret_cast<const bf16x4*>(a.bias + ncol0 + nb * 32 + 8 * g + 4 * hh);
    bf16x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (bf16)(acc[nb][g][e] + (float)b[e]);
    return v;
  });
}

template <int GBM, int SLOTS>
int launch_rows(const GemmArgs& a, const GemmPlan& p, hipStream_t s) {
  const int64_t tiles = ((int64_t)a.M + GBM - 1) / GBM * (a.N / GBN);
  if (tiles > 0x7fffffff) return set_error(2, "gemm: %lld tiles too many", (long long)tiles);
  const dim3 block(64 * kGemmWM * kGemmWN);
  if (p.splits > 1) {
    GemmArgs as = a;
    as.split_from = p.from;
    as.splits = p.splits;
    hipLaunchKernelGGL((gemm_rowsq_kernel<kGemmWM, kGemmWN, kGemmBK, GBM, SLOTS, true>),
                       dim3((unsigned)(p.from + p.rest * p.splits)), block, 0, s, as);
    hipLaunchKernelGGL(gemm_merge_kernel, dim3((unsigned)(p.rest * (GBM / 32))), dim3(256), 0, s, as, GBM);
  } else {
    hipLaunchKernelGGL((gemm_rowsq_kernel<kGemmWM, kGemmWN, kGemmBK, GBM, SLOTS, false>), dim3((unsigned)tiles),
                       block, 0, s, a);
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : set_error(4, "gemm launch: %s", hipGetErrorString(e));
}

}  // namespace

size_t gemm_split_bytes(int M, int N, int K) {
  if (M <= 0 || N < GBN || K < kGemmBK) return 0;
  return gemm_plan_bytes(gemm_plan(M, N, K, K, device_cu_count(), SIZE_MAX));
}

int launch_gemm_rowsq(const GemmArgs& a, hipStream_t s) {
  if (a.M == 0) return 0;
  const GemmPlan p = gemm_plan(a.M, a.N, a.K, a.ldx, device_cu_count(), a.part != nullptr ? a.part_bytes : 0);
  // as many slots as the 160 KB of LDS hold
  switch (p.rows) {
    case 320: return launch_rows<320, 2>(a, p, s);
    case 256: return launch_rows<256, 2>(a, p, s);
    case 192: return launch_rows<192, 2>(a, p, s);
    default: return launch_rows<128, 3>(a, p, s);
  }
}

}  // namespace wan

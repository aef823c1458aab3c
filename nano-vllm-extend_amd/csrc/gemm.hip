// The GDN layer's projections: C = A B^T on the bf16 matrix cores with fp32
// accumulation (F.linear with an nn.Linear weight, nanovllm/layers/linear.py:56-75,
// :133-158; called at nanovllm/models/qwen3_5.py:929-939, :964, :1008-1010,
// :1086).
//
//   A [M, K] bf16, row stride lda (activations: tokens x hidden, or the gated
//     norm's output for out_proj)
//   B [N, K] bf16, row stride ldb (the weight as nn.Linear stores it)
//   C [M, N] bf16, row stride ldc
//
// Both operands are K-contiguous, which is the layout the matrix-core
// fragments want: a 32x32x16 bf16 product takes from each lane 8 consecutive
// k values of one row of each operand, so every operand read is one 16-byte
// LDS read.
//
// Four kernels, chosen by gemm_launch:
//   gemm_tn_pp_kernel    256 x 256 tiles, the last few as 128 x 128 quarters, or
//                        128 x 128 blocks alone; 8 waves in two alternating
//                        groups, persistent (most shapes with more than a few
//                        hundred rows)
//   gemm_tn_ring_kernel  16, 32 or 64 rows x 32 columns, K dealt to the waves,
//                        a load ring per wave (few tiles: a decode out_proj)
//   gemm_tn_deep_kernel  64 x 128 or 64 x 64, three or four LDS stages (a
//                        decode in_proj)
//   gemm_tn_kernel       the general one: 256 x 256 or 192 x 256 where K is an
//                        odd multiple of 64 or 192-row tiles run in one round,
//                        64-row tiles where K is short
// All but the ring kernel add a row's products in K's order, so they give the
// same bits; the ring kernel adds four partial sums.
//
// gemm_tn_kernel: a workgroup of 4 waves (one per SIMD, one workgroup per CU)
// computes a BM x BN tile of C, K in steps of 64.  Wave (wm, wn) owns rows BM /
// 2 wm .. and columns BN / 2 wn ..: BM / 64 x BN / 64 accumulator tiles of 32 x
// 32 (256 registers at 256 x 256, kept in AGPRs), 64 products per step.
//
// Operand path (all kernels): global -> LDS directly (buffer_load ... lds, no
// registers).  gemm_tn_kernel has two stages of BM + BN rows x 128 bytes (128
// KiB at 256 x 256).  The loads
// of step s + 1 are spread one per product over the first half of step s (a
// burst stalls the waves on the shared address unit).  Operand fragments
// are read one 16-deep sub-step ahead of their products, interleaved one read
// per product.  One workgroup barrier per step, placed before the last
// sub-step's products so the next stage's first reads overlap them.  LDS
// rows have their eight 16-byte granules XOR-swizzled by (row / 2) % 8, which
// makes the fragment reads free of bank conflicts (measured: zero).
//
// Tile order: consecutive workgroups run on different XCDs (workgroup b on
// XCD b % 8); the tiles are renumbered so that each XCD walks a contiguous
// range in groups of 4 row blocks x all column blocks, and the tiles resident
// on one XCD at a time share A row blocks and B column blocks in its L2.
//
// Epilogue: the products take B as the first operand, so they are tiles of
// C^T and each lane holds runs of 4 consecutive columns of one row; a lane
// swap (v_permlane32_swap) makes them runs of 8, stored as 16-byte pieces
// straight from the registers.  With gate outputs (GemmGates) the columns
// [gate_col, gate_col + Hv) are the b projection and [gate_col + Hv, gate_col
// + 2 Hv) the a projection: besides their bf16 values, beta = sigmoid(b)
// (bf16) and g = -exp(A_log) softplus(a + dt_bias) (fp32) are written from the
// bf16-rounded values with the gate kernel's arithmetic (gdn::gate_beta,
// gdn::gate_g), so they equal gdn_g_beta applied to C.
#include <algorithm>

#include "gdn_common.h"

namespace {

constexpr int kBK = 64;  // the tile (BM x BN) is a template argument
constexpr int kGemmThreads = 256;
constexpr int kGroupM = 4;  // row blocks per tile group
constexpr int kCUs = gdn::kNumCu;

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// The output: C's columns in up to four parts, part s holding columns
// [end[s - 1], end[s]) (end[-1] = 0) at c[s] with row stride ld[s]; vec[s]: its
// rows take 16-byte stores.  Every part boundary is a multiple of 16, so each
// 16-column half of a 32-column block (one store pair of every lane) lies in
// one part, and the part is the same for the whole wave.
constexpr int kMaxParts = 4;
struct GemmOut {
  uint16_t* c[kMaxParts];
  int64_t ld[kMaxParts];
  int end[kMaxParts];
  int vec[kMaxParts];
};

struct GemmGates {
  float* g;               // [M, Hv] fp32 (NULL: no gate outputs)
  uint16_t* beta;         // [M, Hv] bf16
  const void* A_log;      // [Hv], bf16 or fp32 (param_f32)
  const void* dt_bias;
  int param_f32;
  int gate_col;           // first b column of C
  int Hv;
};

// Byte offset of granule c (16 bytes) of row r in a 128-byte-row LDS tile.
// Granules are XOR-swizzled by (r / 2) % 8: a 16-byte read serves 16 lanes
// at a time from 256 bytes of banks (two rows), and the 16 lanes of a
// fragment read (16 consecutive rows, one granule) then hit 16 distinct
// 16-byte bank groups.
__device__ __forceinline__ int sw_off(int r, int c) { return r * 128 + ((c ^ ((r >> 1) & 7)) << 4); }

__device__ __forceinline__ f32x16_t mfma_bf16(const gdn::s16x8_t& a, const gdn::s16x8_t& b, const f32x16_t& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(gdn::bf16x8_t, a),
                                                 __builtin_bit_cast(gdn::bf16x8_t, b), c, 0, 0, 0);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), static_cast<short>(0), 0x7fffffff, 0x00020000);
}

// Direct-to-LDS loads: one buffer_load_dwordx4 ... lds moves 64 lanes x 16
// bytes into the 1 KiB of LDS at M0 + 16 lane.  A stage holds the A tile (BM
// rows) then the B tile (256 rows), 128 bytes a row: 1 KiB block b is tile rows
// 8 b' .. 8 b' + 7 (b' = b for A, b - BM / 8 for B; BM / 8 is even).  Lane l
// fills row 8 b' + l / 8, slot l % 8, which under the swizzle holds the row's
// global granule (l % 8) ^ (4 (b % 2) + l / 16).  Wave w loads blocks w,
// w + 4, w + 8, ...
typedef __attribute__((address_space(3))) void* lds_ptr_t;

__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rsrc, uint8_t* lds, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)lds, 16, voff, soff, 0, 0);
}

__device__ __forceinline__ f32x16_t zero16() {
  f32x16_t z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.f;
  return z;
}

// Epilogue of a BM x BN tile, straight from the accumulators of wave
// (wm, wn).  `scratch`: (BM / 2) x 32 bf16 per wave of LDS that nothing reads
// any more (the gate outputs go through it).
template <int BM, int BN>
__device__ __forceinline__ void gemm_store(const f32x16_t (&acc)[BM / 64][BN / 64], const GemmOut& out, int M,
                                           int N, int m0, int n0, int wave, int lane, const GemmGates& gt,
                                           uint8_t* scratch) {
  constexpr int MI = BM / 64, NJ = BN / 64;
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 31, lg = lane >> 5;
  // acc[i][j] register 4 q + r of lane (li, lg) is C[row][col + r] with row =
  // m0 + BM / 2 wm + 32 i + li, col = n0 + BN / 2 wn + 32 j + 8 q + 4 lg.  One
  // swap between lanes l and l + 32 (v_permlane32_swap: the upper half of the
  // first operand with the lower half of the second) leaves lane (li, lg)
  // columns 16 p + 8 lg .. + 7 of pair p = (q 2p, q 2p + 1) in bf16: one
  // 16-byte store per pair, two lanes filling 32 bytes of a row.
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int m = m0 + (BM / 2) * wm + 32 * i + li;
    const bool row_ok = m < M;  // (no early exit: the gate loop below spans every lane)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int cb = n0 + (BN / 2) * wn + 32 * j;  // wave-uniform
      if (cb >= N) continue;
      // the output part of this block's first 16 columns (wave-uniform;
      // selects with constant indices, so the part table stays in scalar
      // registers)
      int s = cb < out.end[0] ? 0 : cb < out.end[1] ? 1 : cb < out.end[2] ? 2 : 3;
      auto pick = [&s](auto a0, auto a1, auto a2, auto a3) { return s == 0 ? a0 : s == 1 ? a1 : s == 2 ? a2 : a3; };
      int cbeg = pick(0, out.end[0], out.end[1], out.end[2]);
      int cend = pick(out.end[0], out.end[1], out.end[2], out.end[3]);
      bool vec = pick(out.vec[0], out.vec[1], out.vec[2], out.vec[3]) != 0;
      uint16_t* crow = pick(out.c[0], out.c[1], out.c[2], out.c[3]) +
                       static_cast<int64_t>(row_ok ? m : 0) * pick(out.ld[0], out.ld[1], out.ld[2], out.ld[3]) - cbeg;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        if (p == 1 && cend == cb + 16 && cend < N) {
          // the second 16 columns open the next part (a boundary inside the
          // block: rare)
          ++s;
          cbeg = cend;
          cend = pick(out.end[0], out.end[1], out.end[2], out.end[3]);
          vec = pick(out.vec[0], out.vec[1], out.vec[2], out.vec[3]) != 0;
          crow = pick(out.c[0], out.c[1], out.c[2], out.c[3]) +
                 static_cast<int64_t>(row_ok ? m : 0) * pick(out.ld[0], out.ld[1], out.ld[2], out.ld[3]) - cbeg;
        }
        const int q = 2 * p;
        const auto lo = __builtin_amdgcn_permlane32_swap(gdn::f2bf2(acc[i][j][4 * q], acc[i][j][4 * q + 1]),
                                                         gdn::f2bf2(acc[i][j][4 * q + 4], acc[i][j][4 * q + 5]),
                                                         false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(gdn::f2bf2(acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]),
                                                         gdn::f2bf2(acc[i][j][4 * q + 6], acc[i][j][4 * q + 7]),
                                                         false, false);
        const uint32_t w[4] = {lo[0], hi[0], lo[1], hi[1]};  // columns n .. n + 7
        const int n = cb + 16 * p + 8 * lg;
        if (!row_ok) {
        } else if (vec && n + 8 <= cend) {
          *reinterpret_cast<uint4*>(crow + n) = make_uint4(w[0], w[1], w[2], w[3]);
        } else {
#pragma unroll
          for (int t = 0; t < 8; ++t)
            if (n + t < cend) crow[n + t] = static_cast<uint16_t>(w[t / 2] >> (16 * (t % 2)));
        }
      }
      // Gate outputs from the bf16-rounded b and a columns of this 32-column
      // block.  The block's values go through the wave's own 8 KiB of the
      // stage the last step no longer reads (wave-local, in order), and a
      // rolled loop computes beta and g (unrolled over the registers, the gate
      // arithmetic would not fit beside the accumulators).
      if (gt.g && cb + 32 > gt.gate_col && cb < gt.gate_col + 2 * gt.Hv) {
        uint16_t* gs = reinterpret_cast<uint16_t*>(scratch) + wave * (BM / 2) * 32;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t lo = gdn::f2bf2(acc[i][j][4 * q], acc[i][j][4 * q + 1]);
          const uint32_t hi = gdn::f2bf2(acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
          *reinterpret_cast<uint2*>(gs + 32 * (32 * i + li) + 8 * q + 4 * lg) = make_uint2(lo, hi);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
#pragma unroll 1
        for (int e = lane; e < 32 * 32; e += 64) {
          const int r = e >> 5, c = e & 31;
          const int mm = m - li + r, n = cb + c, col = n - gt.gate_col;
          if (mm >= M || n >= N || col < 0 || col >= 2 * gt.Hv) continue;
          const float v = gdn::bf2f(gs[32 * (32 * i + r) + c]);
          if (col < gt.Hv) {
            gt.beta[static_cast<int64_t>(mm) * gt.Hv + col] = gdn::gate_beta(v);
          } else {
            const int h = col - gt.Hv;
            gt.g[static_cast<int64_t>(mm) * gt.Hv + h] =
                gdn::gate_g(v, gdn::load_param(gt.A_log, h, gt.param_f32), gdn::load_param(gt.dt_bias, h, gt.param_f32));
          }
        }
      }
    }
  }
}

// grid = 8 * ceil(tiles / 8); block = 256 (4 waves, 2 x 2 over the tile).
// Wave (wm, wn) owns rows BM / 2 wm .. and columns BN / 2 wn ..: MI x NJ
// accumulator tiles of 32 x 32 (MI = BM / 64, NJ = BN / 64).  kMinWG
// workgroups per CU bound the registers (1: 512 per lane, AGPRs included).
template <int BM, int BN, int kMinWG>
__global__ __launch_bounds__(kGemmThreads, kMinWG) void gemm_tn_kernel(const uint16_t* __restrict__ A, int64_t lda,
                                                                   const uint16_t* __restrict__ B, int64_t ldb,
                                                                   GemmOut out, int M,
                                                                   int N, int K, GemmGates gt) {
  constexpr int MI = BM / 64, NJ = BN / 64;
  constexpr int kStage = (BM + BN) * 128;  // bytes per stage: 64 KiB at 256 x 256
  constexpr int kPer = (BM + BN) / 32;     // 1 KiB blocks per wave per stage (= 2 (MI + NJ))
  constexpr int kAPer = BM / 32;           // of which A blocks (the first kAPer)
  constexpr int kReads = MI + NJ, kProds = MI * NJ;  // fragment reads, products per sub-step
  constexpr int kPair = kReads < kProds ? kReads : kProds;
  // two stages as two objects, so the compiler sees that products from one
  // do not read what the loads into the other write
  __shared__ __align__(16) uint8_t st0[kStage];
  __shared__ __align__(16) uint8_t st1[kStage];

  const int mb_n = (M + BM - 1) / BM, nb_n = (N + BN - 1) / BN;
  const int64_t tiles = static_cast<int64_t>(mb_n) * nb_n;
  const int64_t L = gdn::xcd_remap(blockIdx.x, tiles);
  if (L < 0) return;
  // tile groups of kGroupM row blocks x all column blocks, row block fastest
  const int64_t per_group = static_cast<int64_t>(kGroupM) * nb_n;
  const int64_t grp = L / per_group, in_grp = L % per_group;
  const int gm = static_cast<int>(min<int64_t>(kGroupM, mb_n - grp * kGroupM));
  const int mb = static_cast<int>(grp * kGroupM + in_grp % gm);
  const int nb = static_cast<int>(in_grp / gm);
  const int m0 = mb * BM, n0 = nb * BN;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 31, lg = lane >> 5;

  // per-lane global byte offsets of the wave's kPer blocks (rows clamped:
  // rows past M (N) re-read the last row; their results are not stored)
  const __amdgpu_buffer_rsrc_t ra = rsrc_of(A), rb = rsrc_of(B);
  int goff[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int b = wave + 4 * i;
    const int gcol = 8 * ((lane & 7) ^ (((b & 1) << 2) | (lane >> 4)));
    if (i < kAPer) {
      goff[i] = static_cast<int>((min(m0 + 8 * b + (lane >> 3), M - 1) * lda + gcol) * 2);
    } else {
      goff[i] = static_cast<int>((min(n0 + 8 * (b - BM / 8) + (lane >> 3), N - 1) * ldb + gcol) * 2);
    }
  }
  const int nk = K / kBK;
  // the wave's blocks i0 .. i0 + n - 1 of step `step` (clamped to the last
  // step: the loads after the last step repeat it into the unused stage)
  auto issue = [&](uint8_t* st, int step, int i0, int n) {
    const int kbyte = min(step, nk - 1) * kBK * 2;
#pragma unroll
    for (int i = i0; i < i0 + n; ++i) dma16(i < kAPer ? ra : rb, st + (wave + 4 * i) * 1024, goff[i], kbyte);
  };

  f32x16_t acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = zero16();

  // Operand fragments of one 16-deep sub-step: MI of A, NJ of B (one 16-byte
  // LDS read each).  Fragments are read one sub-step ahead of their
  // products, so each read has a sub-step of products (512 cycles at 256 x
  // 256) to arrive.
  struct Frag {
    gdn::s16x8_t a[MI], b[NJ];
  };
  auto read_frag = [&](const uint8_t* st, int ks, Frag& f) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
      f.a[i] = *reinterpret_cast<const gdn::s16x8_t*>(st + sw_off((BM / 2) * wm + 32 * i + li, 2 * ks + lg));
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      f.b[j] = *reinterpret_cast<const gdn::s16x8_t*>(st + BM * 128 + sw_off((BN / 2) * wn + 32 * j + li, 2 * ks + lg));
  };
  // B as the first operand: the product is the tile of C^T, so each lane's
  // four consecutive accumulator registers are four consecutive columns of
  // one row of C (stored as one 8-byte piece)
  auto mfmas = [&](const Frag& f) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = mfma_bf16(f.b[j], f.a[i], acc[i][j]);
  };
  // One sub-step's products with the next sub-step's reads between them.
  auto overlap = [&](const Frag& f, const uint8_t* st, int ks, Frag& nf) {
    read_frag(st, ks, nf);
    mfmas(f);
#pragma unroll
    for (int r = 0; r < kPair; ++r) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one product
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read
    }
    if (kProds > kPair) __builtin_amdgcn_sched_group_barrier(0x008, kProds - kPair, 0);
    if (kReads > kPair) __builtin_amdgcn_sched_group_barrier(0x100, kReads - kPair, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  // The same with half of the wave's loads of step `ld` into `dst` as well
  // (kPer / 2 = MI + NJ of them, one after each of the first products).  A
  // burst of loads stalls the wave (the address unit takes 1 KiB per 16
  // cycles, and four waves share it), so they are spread over the products.
  auto overlap_ld = [&](const Frag& f, const uint8_t* st, int ks, Frag& nf, uint8_t* dst, int ld, int i0) {
    read_frag(st, ks, nf);
    issue(dst, ld, i0, kPer / 2);
    mfmas(f);
#pragma unroll
    for (int r = 0; r < kPair; ++r) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one product
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // one load
    }
    if (kProds > kPair) __builtin_amdgcn_sched_group_barrier(0x008, kProds - kPair, 0);
    if (kReads > kPair) {
      __builtin_amdgcn_sched_group_barrier(0x100, kReads - kPair, 0);
      __builtin_amdgcn_sched_group_barrier(0x020, kReads - kPair, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // Step s (4 sub-steps) is multiplied from stage s % 2 while step s + 1 is
  // loaded into the other stage (during its first two sub-steps).  The barrier comes once the step's last
  // fragments are read (before their products): it waits for the wave's own
  // loads first, so after it the next stage is complete for every wave and
  // no wave reads the current stage any more (the loads of step s + 2 may
  // overwrite it).  The next step's first fragments are read behind the last
  // sub-step's products (no branch on the accumulators' path: a branch there
  // makes the compiler copy them and spill).
  Frag f0, f1;
  auto step = [&](uint8_t* cur, uint8_t* nxt, int s) {
    overlap_ld(f0, cur, 1, f1, nxt, s + 1, 0);
    overlap_ld(f1, cur, 2, f0, nxt, s + 1, kPer / 2);
    overlap(f0, cur, 3, f1);
    __syncthreads();
    overlap(f1, nxt, 0, f0);  // after the last step these reads go unused
  };
  issue(st0, 0, 0, kPer);
  __syncthreads();
  read_frag(st0, 0, f0);
  int s = 0;
  for (; s + 1 < nk; s += 2) {
    step(st0, st1, s);
    step(st1, st0, s + 1);
  }
  if (s < nk) step(st0, st1, s);  // the last step when nk is odd
  gemm_store<BM, BN>(acc, out, M, N, m0, n0, wave, lane, gt, nk % 2 ? st0 : st1);
}

// ---- 16 rows x 32 columns of accumulators to the output (the 8-wave kernel) ----
// Lane (lr, lg) holds C[row0 + lr][cb + 8 lg .. + 7] in c0 (the first four) and
// c1: one 16-byte piece, four lanes filling 64 contiguous bytes of a row.
__device__ __forceinline__ void gemm_store16(const gdn::f32x4_t& c0, const gdn::f32x4_t& c1, const GemmOut& out,
                                             int M, int N, int row0, int cb, int lane, const GemmGates& gt,
                                             uint16_t* gs) {
  const int lr = lane & 15, lg = lane >> 4;
  if (cb >= N || row0 >= M) return;  // wave-uniform
  auto pick = [](int t, auto a0, auto a1, auto a2, auto a3) { return t == 0 ? a0 : t == 1 ? a1 : t == 2 ? a2 : a3; };
  const uint4 w = make_uint4(gdn::f2bf2(c0[0], c0[1]), gdn::f2bf2(c0[2], c0[3]), gdn::f2bf2(c1[0], c1[1]),
                             gdn::f2bf2(c1[2], c1[3]));
  // the part of the block's first 16 columns (wave-uniform)
  const int s = cb < out.end[0] ? 0 : cb < out.end[1] ? 1 : cb < out.end[2] ? 2 : 3;
  const int cend = pick(s, out.end[0], out.end[1], out.end[2], out.end[3]);
  const int m = row0 + lr, n = cb + 8 * lg;
  if (pick(s, out.vec[0], out.vec[1], out.vec[2], out.vec[3]) && cb + 32 <= cend) {
    // the whole block in one part with 16-byte rows
    uint16_t* c = pick(s, out.c[0], out.c[1], out.c[2], out.c[3]) - pick(s, 0, out.end[0], out.end[1], out.end[2]);
    const int64_t ld = pick(s, out.ld[0], out.ld[1], out.ld[2], out.ld[3]);
    if (m < M) *reinterpret_cast<uint4*>(c + m * ld + n) = w;
  } else if (m < M) {
    // a part boundary inside the block, the last columns, or rows without
    // 16-byte alignment
    const int sp = n >= cend && cend < N ? s + 1 : s;
    const int pe = pick(sp, out.end[0], out.end[1], out.end[2], out.end[3]);
    const int pb = pick(sp, 0, out.end[0], out.end[1], out.end[2]);
    uint16_t* crow = pick(sp, out.c[0], out.c[1], out.c[2], out.c[3]) +
                     static_cast<int64_t>(m) * pick(sp, out.ld[0], out.ld[1], out.ld[2], out.ld[3]) - pb;
    if (pick(sp, out.vec[0], out.vec[1], out.vec[2], out.vec[3]) && n + 8 <= pe) {
      *reinterpret_cast<uint4*>(crow + n) = w;
    } else {
      const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int t = 0; t < 8; ++t)
        if (n + t < pe) crow[n + t] = static_cast<uint16_t>(ww[t / 2] >> (16 * (t % 2)));
    }
  }
  // gate outputs from the bf16-rounded b and a columns of this block, through
  // the wave's own 1 KiB of LDS (see gemm_store)
  if (gt.g && cb + 32 > gt.gate_col && cb < gt.gate_col + 2 * gt.Hv) {
    *reinterpret_cast<uint4*>(gs + 32 * lr + 8 * lg) = w;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
#pragma unroll 1
    for (int e = lane; e < 16 * 32; e += 64) {
      const int r = e >> 5, c = e & 31;
      const int mm = row0 + r, nn = cb + c, col = nn - gt.gate_col;
      if (mm >= M || nn >= N || col < 0 || col >= 2 * gt.Hv) continue;
      const float v = gdn::bf2f(gs[32 * r + c]);
      if (col < gt.Hv) {
        gt.beta[static_cast<int64_t>(mm) * gt.Hv + col] = gdn::gate_beta(v);
      } else {
        const int h = col - gt.Hv;
        gt.g[static_cast<int64_t>(mm) * gt.Hv + h] =
            gdn::gate_g(v, gdn::load_param(gt.A_log, h, gt.param_f32), gdn::load_param(gt.dt_bias, h, gt.param_f32));
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
  }
}

// ---- 256 x 256 tiles, 8 waves in two alternating groups ----
// What bounds it: the matrix cores at the clock that the power limit leaves
// (8192^3: busy 0.83-0.87 of the cycles at 1.6 GHz).
//
// Two waves per SIMD, one of each group (wave w and w + 4: row halves wm = 0
// and 1).  A K-step of 64 is two load sections (12 LDS fragment reads, 4 loads
// into LDS, a wait) and two product sections (32 products of 16 x 16 x 32: 512
// cycles) per wave, separated by workgroup barriers; group 1 runs one section
// behind group 0, so on each SIMD one wave multiplies while the other reads and
// loads, and neither the address unit nor an LDS wait holds up the products, as
// they do with one wave per SIMD (gemm_tn_kernel).  Sections of 16 products (4
// load sections per step) were slower: 16384 x 12352 x 2048 651 -> 646 us with
// the longer ones, 8192^3 774 -> 757.  Products of 16 x 16 x 32 move half the
// accumulator bytes per operation of 32 x 32 x 16 ones, which the power limit
// turns into clock: 653 -> 613 us and 768 -> 704 us.
//
// LDS: half tiles of 128 rows x 64 values (16 KiB), two of A, two of B, two
// stages; eight objects, so that the compiler's load counting sees which reads
// wait for which loads.  A section loads into the two half tiles that the
// section before it read (both groups are done with them: group 1's reads of
// that section ended before the barrier that started this one), so every load
// has three sections (1,500 cycles and more) to land; the wait at a section's
// end leaves the newest two sections' loads (8) in flight.  The reads of a
// section are: row half 0 of A, column half 1 of B; then row half 1 of A and
// column half 0 of B of the next step (the other column half stays in
// registers).
//
// Persistent: one workgroup per CU walks its tiles, and the loads run on into
// the next tile's first steps, in flight during the stores of this one.  The
// tiles past the last full round of 256 (up to 128 of them) run as quarters of
// 128 x 128 over all CUs: 12.25 rounds cost 12.4 and not 13 (16384 x 12352 x
// 2048: 611 -> 593 us; 2.09 rounds, 17001 x 2048 x 2048: 135 -> 116).
//
// Columns: B's rows are read in the order 8 (j / 4) + 4 t + j % 4 (fragment row
// j of column tile t), so that a lane's two accumulators of a tile pair are 8
// consecutive columns of a row and the stores need no lane exchange; B's LDS
// swizzle follows that order (swb_off).
//
// Against the one-wave-per-SIMD kernel, same box: 16384 x 12352 x 2048 760 ->
// 593 us (1.40 PFLOP/s), 16384 x 2048 x 4096 206 -> 185, 17001 x 8224 x 2048
// 508 -> 425, 1949 x 12352 x 2048 100 -> 87, 1949 x 2048 x 4096 42.6 -> 38.
constexpr int kPPThreads = 512;

__device__ __forceinline__ void half_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}

// s_waitcnt vmcnt(8) lgkmcnt(0): all but the newest 8 loads have landed and
// every LDS read has returned
constexpr int kWaitPP = 8 | (7 << 4);
// s_waitcnt lgkmcnt(0) alone (vmcnt 63)
constexpr int kWaitLds = 15 | (7 << 4) | (3 << 14);

// LDS offset of granule c of row r in a half tile of B (see the column order
// below)
__device__ __forceinline__ int swb_off(int r, int c) {
  return r * 128 + ((c ^ (((r >> 1) & 1) | (((r >> 3) & 3) << 1))) << 4);
}

// grid = 8 * min(32, ...) workgroups of 512; tiles 0 .. whole - 1 run as 256 x
// 256, the rest as quarters.  K is a multiple of 128.
__global__ __launch_bounds__(kPPThreads, 2) void gemm_tn_pp_kernel(const uint16_t* __restrict__ A, int64_t lda,
                                                                  const uint16_t* __restrict__ B, int64_t ldb,
                                                                  GemmOut out, int M, int N, int K, GemmGates gt,
                                                                  int whole) {
  constexpr int kHalf = 128 * 128;  // bytes of a half tile: 128 rows of 64 values
  __shared__ __align__(16) uint8_t a00[kHalf];
  __shared__ __align__(16) uint8_t a01[kHalf];
  __shared__ __align__(16) uint8_t a10[kHalf];
  __shared__ __align__(16) uint8_t a11[kHalf];
  __shared__ __align__(16) uint8_t b00[kHalf];
  __shared__ __align__(16) uint8_t b01[kHalf];
  __shared__ __align__(16) uint8_t b10[kHalf];
  __shared__ __align__(16) uint8_t b11[kHalf];
  __shared__ __align__(16) uint16_t gscr[8][16 * 32];

  const int mb_n = (M + 255) / 256, nb_n = (N + 255) / 256;
  // XCD x (workgroups b % 8 == x) walks a contiguous range of the tiles
  const int xcd = blockIdx.x % gdn::kNumXcd, slot = blockIdx.x / gdn::kNumXcd, stride = gridDim.x / gdn::kNumXcd;
  const int tiles = mb_n * nb_n;
  const int per_xcd = (whole + gdn::kNumXcd - 1) / gdn::kNumXcd;
  const int xend = min((xcd + 1) * per_xcd, whole);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int lr = lane & 15, lg = lane >> 4;

  auto tile_of = [&](int t, int& m0, int& n0) {
    const int per_group = kGroupM * nb_n;
    const int grp = t / per_group, in_grp = t % per_group;
    const int gm = min(kGroupM, mb_n - grp * kGroupM);
    m0 = 256 * (grp * kGroupM + in_grp % gm);
    n0 = 256 * (in_grp / gm);
  };
  // the wave's loads: 1 KiB blocks w and w + 8 of each half tile
  const __amdgpu_buffer_rsrc_t ra = rsrc_of(A), rb = rsrc_of(B);
  const int ldrow = 8 * wave + (lane >> 3);
  const int gcol_a = 8 * ((lane & 7) ^ (((wave & 1) << 2) | (lane >> 4)));
  const int gcol_b = 8 * ((lane & 7) ^ (((wave & 3) << 1) | ((lane >> 4) & 1)));
  int va[2][2], vb[2][2];
  auto set_offsets = [&](int m0, int n0) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        va[h][i] = static_cast<int>((min(m0 + 128 * h + 64 * i + ldrow, M - 1) * lda + gcol_a) * 2);
        vb[h][i] = static_cast<int>((min(n0 + 128 * h + 64 * i + ldrow, N - 1) * ldb + gcol_b) * 2);
      }
  };
  auto dma = [&](const __amdgpu_buffer_rsrc_t& r, uint8_t* dst, const int (&v)[2], int kbyte) {
#pragma unroll
    for (int i = 0; i < 2; ++i) dma16(r, dst + (wave + 8 * i) * 1024, v[i], kbyte);
  };
  typedef gdn::s16x8_t frag_t;
  auto read_a = [&](const uint8_t* h, frag_t (&f)[4][2]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        f[i][ks] = *reinterpret_cast<const frag_t*>(h + sw_off(64 * wm + 16 * i + lr, 4 * ks + lg));
  };
  auto read_b = [&](const uint8_t* h, frag_t (&f)[2][2]) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        f[t][ks] = *reinterpret_cast<const frag_t*>(h + swb_off(32 * wn + 8 * (lr >> 2) + 4 * t + (lr & 3), 4 * ks + lg));
  };
  gdn::f32x4_t acc[2][2][4][2];  // [row half][column half][16-row tile][column tile]
  // one row half of A against both column halves of B
  auto prod = [&](gdn::f32x4_t (&c0)[4][2], gdn::f32x4_t (&c1)[4][2], const frag_t (&fa)[4][2],
                  const frag_t (&f0)[2][2], const frag_t (&f1)[2][2]) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < 2; ++t) c0[i][t] = gdn::mfma16x16x32(f0[t][ks], fa[i][ks], c0[i][t]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < 2; ++t) c1[i][t] = gdn::mfma16x16x32(f1[t][ks], fa[i][ks], c1[i][t]);
    }
    __builtin_amdgcn_s_setprio(0);
    half_barrier();
  };
  auto mem_end = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kWaitPP);
    half_barrier();
  };
  const int nk = K / kBK;  // even
  int L = xcd * per_xcd + slot;
  if (L < xend) {
  int m0, n0;
  tile_of(L, m0, n0);
  set_offsets(m0, n0);
  dma(rb, b00, vb[0], 0);
  dma(ra, a00, va[0], 0);
  dma(rb, b01, vb[1], 0);
  dma(rb, b10, vb[0], 128);
  dma(ra, a01, va[1], 0);
  dma(ra, a10, va[0], 128);
  dma(rb, b11, vb[1], 128);
  frag_t fa[4][2], fb0[2][2], fb1[2][2], fbn[2][2];
  __builtin_amdgcn_s_waitcnt(12 | (7 << 4));
  half_barrier();
  read_b(b00, fb0);
  mem_end();
  for (;;) {
    const int Ln = L + stride;
    const int m0c = m0, n0c = n0;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int t = 0; t < 2; ++t) acc[a][b][i][t] = gdn::f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (wm) half_barrier();
    int kb = 256;
    for (int s = 0; s < nk; s += 2) {
      const int ka = kb - 128;  // of step s + 1: the current tile's
      int v1[2] = {va[1][0], va[1][1]};
      if (s + 2 == nk) {
        // the next loads are the next tile's first steps (past the last tile
        // they repeat this one's)
        if (Ln < xend) {
          tile_of(Ln, m0, n0);
          set_offsets(m0, n0);
        }
        kb = 0;
      }
      dma(rb, b00, vb[0], kb);
      dma(ra, a11, v1, ka);
      read_a(a00, fa);
      read_b(b01, fb1);
      mem_end();
      prod(acc[0][0], acc[0][1], fa, fb0, fb1);
      dma(ra, a00, va[0], kb);
      dma(rb, b01, vb[1], kb);
      read_a(a01, fa);
      read_b(b10, fbn);
      mem_end();
      prod(acc[1][0], acc[1][1], fa, fb0, fb1);
      dma(rb, b10, vb[0], kb + 128);
      dma(ra, a01, va[1], kb);
      read_a(a10, fa);
      read_b(b11, fb1);
      mem_end();
      prod(acc[0][0], acc[0][1], fa, fbn, fb1);
      dma(ra, a10, va[0], kb + 128);
      dma(rb, b11, vb[1], kb + 128);
      read_a(a11, fa);
      read_b(b00, fb0);
      mem_end();
      prod(acc[1][0], acc[1][1], fa, fbn, fb1);
      kb += 256;
    }
    if (!wm) half_barrier();
    // (the lane from an opaque copy, so that no address of the epilogue is
    // kept in registers across the loop)
    int tid_e = static_cast<int>(threadIdx.x);
    asm volatile("" : "+v"(tid_e));
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          gemm_store16(acc[a][b][i][0], acc[a][b][i][1], out, M, N, m0c + 128 * a + 64 * wm + 16 * i,
                       n0c + 128 * b + 32 * wn, tid_e & 63, gt, gscr[wave]);
    if (Ln >= xend) break;
    L = Ln;
  }
  }
  // The tiles after the whole ones, as quarters of 128 x 128: per K-step one
  // half tile of A and one of B, so the eight LDS objects hold four steps.
  // Without whole tiles they are the 128 x 128 blocks of C, in groups of as many
  // rows: the quarters of 256 x 256 tiles that lie past M or N would take
  // workgroups' turns (300 x 8224: 195 blocks in 264 quarters, two turns for some
  // workgroups and none for others, 35.6 us at K = 2048; in blocks 21.1).
  const int mq_n = (M + 127) / 128, nq_n = (N + 127) / 128;
  const int nq = whole ? 4 * (tiles - whole) : mq_n * nq_n;
  const int q_xcd = (nq + gdn::kNumXcd - 1) / gdn::kNumXcd;
  const int qend = min((xcd + 1) * q_xcd, nq);
  for (int q = xcd * q_xcd + slot; q < qend; q += stride) {
    int m0, n0;
    if (whole) {
      tile_of(whole + (q >> 2), m0, n0);
      m0 += 128 * ((q >> 1) & 1);
      n0 += 128 * (q & 1);
      if (m0 >= M || n0 >= N) continue;  // (the whole workgroup)
    } else {
      const int per_group = 2 * kGroupM * nq_n;
      const int grp = q / per_group, in_grp = q % per_group;
      const int gm = min(2 * kGroupM, mq_n - grp * 2 * kGroupM);
      m0 = 128 * (grp * 2 * kGroupM + in_grp % gm);
      n0 = 128 * (in_grp / gm);
    }
    set_offsets(m0, n0);
    __builtin_amdgcn_s_waitcnt(7 << 4);  // loads into the stages, of a tile before
    half_barrier();
    auto load = [&](uint8_t* a, uint8_t* b, int step) {
      const int kb = 128 * min(step, nk - 1);
      dma(ra, a, va[0], kb);
      dma(rb, b, vb[0], kb);
    };
    load(a00, b00, 0);
    load(a01, b01, 1);
    load(a10, b10, 2);
    gdn::f32x4_t c[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < 2; ++t) c[i][t] = gdn::f32x4_t{0.f, 0.f, 0.f, 0.f};
    frag_t fa[4][2], fb[2][2];
    // step s from (a, b); the loads of step s + 3 into (an, bn)
    auto step = [&](const uint8_t* a, const uint8_t* b, uint8_t* an, uint8_t* bn, int s) {
      load(an, bn, s + 3);
      read_a(a, fa);
      read_b(b, fb);
      mem_end();
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int t = 0; t < 2; ++t) c[i][t] = gdn::mfma16x16x32(fb[t][ks], fa[i][ks], c[i][t]);
      __builtin_amdgcn_s_setprio(0);
      half_barrier();
    };
    __builtin_amdgcn_s_waitcnt(kWaitPP);  // step 0
    half_barrier();
    if (wm) half_barrier();
    for (int s = 0; s < nk; s += 4) {
      step(a00, b00, a11, b11, s);
      step(a01, b01, a00, b00, s + 1);
      if (s + 2 >= nk) break;
      step(a10, b10, a01, b01, s + 2);
      step(a11, b11, a10, b10, s + 3);
    }
    if (!wm) half_barrier();
#pragma unroll
    for (int i = 0; i < 4; ++i)
      gemm_store16(c[i][0], c[i][1], out, M, N, m0 + 64 * wm + 16 * i, n0 + 32 * wn, lane, gt, gscr[wave]);
  }
  __builtin_amdgcn_s_waitcnt(0);
}

// ---- few tiles (the out projection of a decode batch): a ring per wave ----
// What bounds it: the loads' latency times the bytes in flight.  Workgroup: BM
// rows x 32 columns of C; the K-steps of 64 are dealt to its four waves in turn
// (wave w: steps w, w + 4, ...), each wave loading its steps into a ring of three
// stages of its own in LDS, so the loop has no barrier and up to 144 KiB per CU
// are in flight.  The waves' partial sums are added through LDS in wave order.
// (Operands loaded straight to registers instead, 16 rows x 64 bytes per load:
// 1 x 2048 x 4096 14.8 us, 64 x 12352 x 2048 24-75 us against 11; the address
// unit pays per row.)  Against the 64 x 64 deep kernel: 1 x 2048 x 4096 16.8 ->
// 6.2 us, 64 rows 17.1 -> 7.9, 200 rows 17.2 -> 11.7; 256 x 2048 x 2048 10.5 ->
// 8.1.
template <int BM>
__global__ __launch_bounds__(kGemmThreads) void gemm_tn_ring_kernel(const uint16_t* __restrict__ A, int64_t lda,
                                                                    const uint16_t* __restrict__ B, int64_t ldb,
                                                                    GemmOut out, int M, int N, int K, GemmGates gt) {
  constexpr int NW = kGemmThreads / 64, NS = 3;
  constexpr int MT = BM / 16, BN = 32;
  constexpr int kStage = (BM + BN) * 128;   // one wave's stage
  constexpr int kPer = (BM + BN) / 8;       // 1 KiB blocks of it
  // s_waitcnt vmcnt: the oldest stage has landed, the loads of the NS - 1 newer
  // ones stay in flight (lgkmcnt 15: no wait)
  constexpr int kVm = (NS - 1) * kPer;
  static_assert(kVm < 64, "vmcnt field");
  constexpr int kWait = (kVm & 15) | (7 << 4) | (15 << 8) | ((kVm >> 4) << 14);
  typedef gdn::s16x8_t frag_t;
  __shared__ __align__(16) uint8_t st0[NW * kStage];
  __shared__ __align__(16) uint8_t st1[NW * kStage];
  __shared__ __align__(16) uint8_t st2[NW * kStage];
  __shared__ __align__(16) uint16_t gscr[NW][16 * 32];
  static_assert(MT * 2048 <= kStage, "the partial sums fit a stage");
  const int mb_n = (M + BM - 1) / BM, nb_n = (N + BN - 1) / BN;
  // the row blocks of a column block on one XCD, so that its L2 reads the weights once
  const int64_t L = gdn::xcd_remap(blockIdx.x, static_cast<int64_t>(mb_n) * nb_n);
  if (L < 0) return;
  const int m0 = BM * static_cast<int>(L % mb_n), n0 = BN * static_cast<int>(L / mb_n);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const __amdgpu_buffer_rsrc_t ra = rsrc_of(A), rb = rsrc_of(B);
  int goff[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    if (i < BM / 8) {
      const int gcol = 8 * ((lane & 7) ^ (((i & 1) << 2) | (lane >> 4)));
      goff[i] = static_cast<int>((min(m0 + 8 * i + (lane >> 3), M - 1) * lda + gcol) * 2);
    } else {
      const int b = i - BM / 8;
      const int gcol = 8 * ((lane & 7) ^ (((b & 3) << 1) | ((lane >> 4) & 1)));
      goff[i] = static_cast<int>((min(n0 + 8 * b + (lane >> 3), N - 1) * ldb + gcol) * 2);
    }
  }
  const int nk = K / kBK;
  auto issue = [&](uint8_t* st, int step) {
    const int kbyte = 128 * min(step, nk - 1);
#pragma unroll
    for (int i = 0; i < kPer; ++i) dma16(i < BM / 8 ? ra : rb, st + wave * kStage + i * 1024, goff[i], kbyte);
  };
  gdn::f32x4_t acc[MT][2];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int t = 0; t < 2; ++t) acc[i][t] = gdn::f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto one = [&](uint8_t* st, int step) {
    const uint8_t* a = st + wave * kStage;
    const uint8_t* b = a + BM * 128;
    frag_t fa[2][MT], fb[2][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
        fa[ks][i] = *reinterpret_cast<const frag_t*>(a + sw_off(16 * i + lr, 4 * ks + lg));
#pragma unroll
      for (int t = 0; t < 2; ++t)
        fb[ks][t] = *reinterpret_cast<const frag_t*>(b + swb_off(8 * (lr >> 2) + 4 * t + (lr & 3), 4 * ks + lg));
    }
    // the reads have returned before the stage is loaded again
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kWaitLds);
    __builtin_amdgcn_sched_barrier(0);
    issue(st, step + NS * NW);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[i][t] = gdn::mfma16x16x32(fb[ks][t], fa[ks][i], acc[i][t]);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kWait);
    __builtin_amdgcn_sched_barrier(0);
  };
  issue(st0, wave);
  issue(st1, wave + NW);
  issue(st2, wave + 2 * NW);
  __builtin_amdgcn_s_waitcnt(kWait);
  int s = wave;
  for (; s + (NS - 1) * NW < nk; s += NS * NW) {
    one(st0, s);
    one(st1, s + NW);
    one(st2, s + 2 * NW);
  }
  if (s < nk) one(st0, s);
  if (s + NW < nk) one(st1, s + NW);
  // the repeated loads past the last step land before the stages are reused
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  gdn::f32x4_t* red = reinterpret_cast<gdn::f32x4_t*>(st0);  // [wave][row tile][column tile][lane]
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int t = 0; t < 2; ++t) red[((wave * MT + i) * 2 + t) * 64 + lane] = acc[i][t];
  __syncthreads();
  for (int i = wave; i < MT; i += NW) {
    gdn::f32x4_t c0 = red[(i * 2) * 64 + lane], c1 = red[(i * 2 + 1) * 64 + lane];
#pragma unroll
    for (int w = 1; w < NW; ++w) {
      c0 += red[((w * MT + i) * 2) * 64 + lane];
      c1 += red[((w * MT + i) * 2 + 1) * 64 + lane];
    }
    gemm_store16(c0, c1, out, M, N, m0 + 16 * i, n0, lane, gt, gscr[wave]);
  }
}

// ---- small M (decode batches): a deeper load pipeline ----
// gemm_tn_kernel's two stages let a step's loads arrive during one step's
// products, which at 64-row tiles are four to eight products: every step then
// waits out the memory latency (its barrier drains every load).  Here the
// tile is 64 x BN and there are NS stages (3 or 4, separate LDS objects): the
// loads of step s + NS - 1 go out at the start of step s, and the barrier
// before step s waits only for the wave's loads of step s (vmcnt down to the
// NS - 2 later steps' loads) and for its own LDS reads (so every wave is done
// with the stage the next loads go into).  Same LDS layout, fragment reads,
// products in the same order and epilogue as gemm_tn_kernel: the results are
// the same bits.  Steps past the last one repeat its loads into the unused
// stages (every path issues the same loads), drained before the epilogue.
// (Graph-replayed, without an exit inside a loop trip: 37 x 12352 x 2048 11.2
// -> 10.5 us, 128 rows 15.2 -> 14.4, 200 rows 21.9 -> 21.3.)
template <int BN, int NS>
__global__ __launch_bounds__(kGemmThreads, 2) void gemm_tn_deep_kernel(const uint16_t* __restrict__ A, int64_t lda,
                                                                    const uint16_t* __restrict__ B, int64_t ldb,
                                                                    GemmOut out, int M,
                                                                    int N, int K, GemmGates gt) {
  static_assert(NS == 3 || NS == 4, "three or four stages");
  constexpr int BM = 64, MI = 1, NJ = BN / 64;
  constexpr int kStage = (BM + BN) * 128;
  constexpr int kPer = (BM + BN) / 32;  // 1 KiB blocks per wave per stage
  constexpr int kAPer = BM / 32;
  // s_waitcnt: vmcnt = the NS - 2 later steps' loads (bits 3:0 and 15:14),
  // expcnt 7 (no wait), lgkmcnt 0
  constexpr int kVm = (NS - 2) * kPer;
  static_assert(kVm < 64, "vmcnt field");
  constexpr int kWait = (kVm & 15) | (7 << 4) | ((kVm >> 4) << 14);
  __shared__ __align__(16) uint8_t st0[kStage];
  __shared__ __align__(16) uint8_t st1[kStage];
  __shared__ __align__(16) uint8_t st2[kStage];
  __shared__ __align__(16) uint8_t st3[NS == 4 ? kStage : 16];

  const int mb_n = (M + BM - 1) / BM, nb_n = (N + BN - 1) / BN;
  const int64_t tiles = static_cast<int64_t>(mb_n) * nb_n;
  const int64_t L = gdn::xcd_remap(blockIdx.x, tiles);
  if (L < 0) return;
  const int64_t per_group = static_cast<int64_t>(kGroupM) * nb_n;
  const int64_t grp = L / per_group, in_grp = L % per_group;
  const int gm = static_cast<int>(min<int64_t>(kGroupM, mb_n - grp * kGroupM));
  const int mb = static_cast<int>(grp * kGroupM + in_grp % gm);
  const int nb = static_cast<int>(in_grp / gm);
  const int m0 = mb * BM, n0 = nb * BN;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 31, lg = lane >> 5;

  const __amdgpu_buffer_rsrc_t ra = rsrc_of(A), rb = rsrc_of(B);
  int goff[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int b = wave + 4 * i;
    const int gcol = 8 * ((lane & 7) ^ (((b & 1) << 2) | (lane >> 4)));
    if (i < kAPer) {
      goff[i] = static_cast<int>((min(m0 + 8 * b + (lane >> 3), M - 1) * lda + gcol) * 2);
    } else {
      goff[i] = static_cast<int>((min(n0 + 8 * (b - BM / 8) + (lane >> 3), N - 1) * ldb + gcol) * 2);
    }
  }
  const int nk = K / kBK;
  auto issue = [&](uint8_t* st, int step) {
    const int kbyte = min(step, nk - 1) * kBK * 2;
#pragma unroll
    for (int i = 0; i < kPer; ++i) dma16(i < kAPer ? ra : rb, st + (wave + 4 * i) * 1024, goff[i], kbyte);
  };

  f32x16_t acc[MI][NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) acc[0][j] = zero16();

  // one step from stage `cur`: the four sub-steps' fragments, then their products
  auto run = [&](const uint8_t* cur) {
    gdn::s16x8_t fa[4], fb[4][NJ];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      fa[ks] = *reinterpret_cast<const gdn::s16x8_t*>(cur + sw_off(32 * wm + li, 2 * ks + lg));
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        fb[ks][j] = *reinterpret_cast<const gdn::s16x8_t*>(cur + BM * 128 +
                                                           sw_off((BN / 2) * wn + 32 * j + li, 2 * ks + lg));
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[0][j] = mfma_bf16(fb[ks][j], fa[ks], acc[0][j]);
  };
  // step s from `cur`, the loads of step s + NS - 1 into `nxt` (the stage of
  // step s - 1, which every wave has finished reading at the barrier)
  auto one = [&](const uint8_t* cur, uint8_t* nxt, int step) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kWait);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    issue(nxt, step + NS - 1);
    __builtin_amdgcn_sched_barrier(0);
    run(cur);
  };
  issue(st0, 0);
  issue(st1, 1);
  if constexpr (NS == 4) issue(st2, 2);
  // (no exit inside a trip: with one, the compiler's load counting merges its
  // states at the loop head and waits there for loads that are meant to stay
  // in flight)
  int s = 0;
  if constexpr (NS == 4) {
    for (; s + 3 < nk; s += 4) {
      one(st0, st3, s);
      one(st1, st0, s + 1);
      one(st2, st1, s + 2);
      one(st3, st2, s + 3);
    }
    if (s < nk) one(st0, st3, s);
    if (s + 1 < nk) one(st1, st0, s + 1);
    if (s + 2 < nk) one(st2, st1, s + 2);
  } else {
    for (; s + 2 < nk; s += 3) {
      one(st0, st2, s);
      one(st1, st0, s + 1);
      one(st2, st1, s + 2);
    }
    if (s < nk) one(st0, st2, s);
    if (s + 1 < nk) one(st1, st0, s + 1);
  }
  // the repeated loads land before a stage is reused as the gates' scratch
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  gemm_store<BM, BN>(acc, out, M, N, m0, n0, wave, lane, gt, st0);
}

}  // namespace

namespace {

// Tile choice and launch for C = A B^T into `out` (arguments checked by the
// entry points).
int gemm_launch(const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb, const GemmOut& out, int M, int N,
                int K, const GemmGates& gt, void* stream) {
  const int64_t nb256 = (N + 255) / 256;
  const int64_t t256 = ((M + 255) / 256) * nb256, t192 = ((M + 191) / 192) * nb256;
  const int64_t t128 = static_cast<int64_t>((M + 127) / 128) * ((N + 127) / 128);
  const int64_t t64x128 = static_cast<int64_t>((M + 63) / 64) * ((N + 127) / 128);
  const int64_t t64 = static_cast<int64_t>((M + 63) / 64) * ((N + 63) / 64);
  const hipStream_t st = static_cast<hipStream_t>(stream);
  auto grid = [](int64_t wgs) {
    return dim3(static_cast<unsigned>(gdn::kNumXcd * ((wgs + gdn::kNumXcd - 1) / gdn::kNumXcd)));
  };
  const dim3 b3(kGemmThreads);
  // The 8-wave kernel (K in pairs of steps) when its 256 x 256 tiles fill half of
  // the CUs, except where 192 x 256 tiles run in one round as well and there are
  // few of them, or as few as the 256-row ones, or K is short: the round is then
  // its rows' time, and the persistent kernel's start is not made up for (900 x
  // 8224 x 2048: 43.6 us against 41.5 with 192 rows, 257 x 32768 52.0 / 45.6, 3000
  // x 3000 45.5 / 42.1; 1200 x 8224 44.1 / 45.2; 1200 x 8224 x 512 16.9 / 16.1).
  const bool wide = t256 >= kCUs / 2;
  const bool one192 = t256 > kCUs / 2 && t192 <= kCUs &&
                      (5 * t192 <= 4 * kCUs || t192 == t256 || K < 16 * kBK);
  // Fewer tiles: as 128 x 128 blocks in one round.  Against 64 x 128 tiles, two of
  // them per CU, they take as long for a few blocks as for 256, so these must have
  // work for more than one tile per CU, few blocks that are half empty, and a K
  // that makes up for the start (1949 x 2048 x 4096: 42.6 -> 37.7 us, 900 x 4096 x
  // 2048 23.9 -> 22.4, 384 x 8224 x 2048 22.2 -> 22.0; the other way 129 x 8224 x
  // 2048 14.4 -> 19.5, 257 x 6144 15.6 -> 20.6, 768 x 4096 x 1024 11.9 -> 12.7, 900 x
  // 4096 x 512 7.7 -> 9.7; two rounds of blocks, 400 x 12352 x 2048 35.0 -> 38.1).
  const bool blocks = !wide && t128 <= kCUs && t64x128 > kCUs && 2 * t64x128 > 3 * t128 &&
                      K * t64x128 >= 1600 * kCUs;
  if (K % (2 * kBK) == 0 && (wide ? !one192 : blocks)) {
    const int64_t rem = t256 % kCUs;
    const int64_t whole = rem <= kCUs / 2 ? t256 - rem : t256;
    const int64_t wgs = std::min<int64_t>(kCUs, whole ? std::max(whole, 4 * (t256 - whole)) : t128);
    gemm_tn_pp_kernel<<<grid(wgs), dim3(kPPThreads), 0, st>>>(A, lda, B, ldb, out, M, N, K, gt,
                                                              static_cast<int>(whole));
    return gdn_launch_status();
  }
  if (wide) {
    // Odd multiples of 64, and one round of 192-row tiles: a launch runs in
    // ceil(tiles / CUs) waves of tiles, each taking time in proportion to the
    // tile's rows; 192 x 256 is taken when its waves x rows is smaller (a short
    // last wave of 256-row tiles, e.g. 536 tiles = 2.09 waves -> 712 = 2.78).
    const int64_t w256 = (t256 + kCUs - 1) / kCUs, w192 = (t192 + kCUs - 1) / kCUs;
    if (w192 * 192 < w256 * 256)
      gemm_tn_kernel<192, 256, 1><<<grid(t192), b3, 0, st>>>(A, lda, B, ldb, out, M, N, K, gt);
    else
      gemm_tn_kernel<256, 256, 1><<<grid(t256), b3, 0, st>>>(A, lda, B, ldb, out, M, N, K, gt);
    return gdn_launch_status();
  }
  // Small M.  The deeper load pipelines pay when K has at least 16 steps (with
  // fewer their prologue and the repeated last loads cost more than they save:
  // 1000 x 2080 x 512: 6.5 -> 7.0 us).
  const bool deep = K / kBK >= 16;
  // Ring tiles of 16, 32 or 64 rows x 32 columns, the smallest with at most one
  // workgroup per CU (with more, the 64-row tiles below move fewer bytes: 64 x
  // 12352 x 2048 11.2 us against 16-19; 500 x 2048 x 2048 13.7 against 13.9), and
  // not 64 rows of an A that is tall and more than the 4 MiB of an XCD's L2: every
  // XCD reads all of A for its column blocks (2000 x 256 x 2048 13.5 us against
  // 9.9 with 64 x 64 tiles, 6000 x 64 x 2048 11.4 / 9.6; 1024 x 512 x 2048 9.2 /
  // 9.9, 1700 x 256 x 1024 6.2 / 6.6; one column block, 16384 x 32 x 1024, 6.3 / 9.0).
  int rows = 16;
  const int64_t nb32 = (N + 31) / 32;
  while (rows <= 64 && (M + rows - 1) / rows * nb32 > kCUs) rows *= 2;
  const bool tall = M > 1024 && N > 32 && static_cast<int64_t>(M) * K > (1 << 21);
  if (deep && rows <= (tall ? 32 : 64)) {
    const dim3 gr = grid((M + rows - 1) / rows * nb32);
    if (rows == 16)
      gemm_tn_ring_kernel<16><<<gr, b3, 0, st>>>(A, lda, B, ldb, out, M, N, K, gt);
    else if (rows == 32)
      gemm_tn_ring_kernel<32><<<gr, b3, 0, st>>>(A, lda, B, ldb, out, M, N, K, gt);
    else
      gemm_tn_ring_kernel<64><<<gr, b3, 0, st>>>(A, lda, B, ldb, out, M, N, K, gt);
    return gdn_launch_status();
  }
  // 64 x 128 tiles, two or more workgroups per CU, spread the work over the
  // whole chip; 64 x 64 when even those would not.
  if (t64x128 >= kCUs / 2) {
    if (deep)
      gemm_tn_deep_kernel<128, 3><<<grid(t64x128), b3, 0, st>>>(A, lda, B, ldb, out, M, N, K, gt);
    else
      gemm_tn_kernel<64, 128, 2><<<grid(t64x128), b3, 0, st>>>(A, lda, B, ldb, out, M, N, K, gt);
  } else {
    if (deep)
      gemm_tn_deep_kernel<64, 4><<<grid(t64), b3, 0, st>>>(A, lda, B, ldb, out, M, N, K, gt);
    else
      gemm_tn_kernel<64, 64, 2><<<grid(t64), b3, 0, st>>>(A, lda, B, ldb, out, M, N, K, gt);
  }
  return gdn_launch_status();
}

// The checks both entry points share: K in steps of 64; 16-byte row pieces
// of A and B; 32-bit buffer offsets; the gate outputs' arguments.
int gemm_check(const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb, int M, int N, int K, float* g,
               uint16_t* beta, const void* A_log, const void* dt_bias, int gate_col, int Hv) {
  if (K % kBK || K == 0 || lda % 8 || ldb % 8 || lda < K || ldb < K || reinterpret_cast<uintptr_t>(A) % 16 ||
      reinterpret_cast<uintptr_t>(B) % 16 || static_cast<int64_t>(M) * lda * 2 >= (1LL << 31) ||
      static_cast<int64_t>(N) * ldb * 2 >= (1LL << 31))
    return GDN_ERR_INVALID_ARG;
  if (g && (!beta || !A_log || !dt_bias || Hv <= 0 || gate_col < 0 || gate_col + 2 * Hv > N)) return GDN_ERR_INVALID_ARG;
  return GDN_OK;
}

// One output part: rows of ld elements at c (16-byte stores when ld is a
// multiple of 8 and c 16-byte aligned, else element by element: c then only
// 2-byte aligned).
bool part_ok(const uint16_t* c, int64_t ld, int width) {
  return c && ld >= width && reinterpret_cast<uintptr_t>(c) % (ld % 8 ? 2 : 16) == 0;
}

}  // namespace

extern "C" int gdn_gemm_bf16(const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb, uint16_t* C,
                             int64_t ldc, int M, int N, int K, float* g, uint16_t* beta, const void* A_log,
                             const void* dt_bias, int param_is_fp32, int gate_col, int Hv, void* stream) {
  if (M < 0 || N < 0 || K < 0) return GDN_ERR_INVALID_ARG;
  if (M == 0 || N == 0) return GDN_OK;
  if (!A || !B || !C) return GDN_ERR_INVALID_ARG;
  const int st = gemm_check(A, lda, B, ldb, M, N, K, g, beta, A_log, dt_bias, gate_col, Hv);
  if (st != GDN_OK) return st;
  if (!part_ok(C, ldc, N)) return GDN_ERR_INVALID_ARG;
  const int v = ldc % 8 == 0;
  const GemmOut out{{C, C, C, C}, {ldc, ldc, ldc, ldc}, {N, N, N, N}, {v, v, v, v}};
  const GemmGates gt{g, beta, A_log, dt_bias, param_is_fp32 ? 1 : 0, gate_col, Hv};
  return gemm_launch(A, lda, B, ldb, out, M, N, K, gt, stream);
}

extern "C" int gdn_gemm_bf16_cols(const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb, int M, int N, int K,
                                  int n_parts, uint16_t* const* C, const int64_t* ldc, const int* col_end, float* g,
                                  uint16_t* beta, const void* A_log, const void* dt_bias, int param_is_fp32,
                                  int gate_col, int Hv, void* stream) {
  if (M < 0 || N < 0 || K < 0 || n_parts < 1 || n_parts > kMaxParts || !C || !ldc || !col_end)
    return GDN_ERR_INVALID_ARG;
  if (M == 0 || N == 0) return GDN_OK;
  if (!A || !B) return GDN_ERR_INVALID_ARG;
  const int st = gemm_check(A, lda, B, ldb, M, N, K, g, beta, A_log, dt_bias, gate_col, Hv);
  if (st != GDN_OK) return st;
  GemmOut out{};
  int beg = 0;
  for (int s = 0; s < kMaxParts; ++s) {
    const int e = s < n_parts ? col_end[s] : N;
    if (s < n_parts) {
      // increasing boundaries at multiples of 16, the last one at N
      if (e <= beg || (s + 1 < n_parts ? e % 16 != 0 || e >= N : e != N)) return GDN_ERR_INVALID_ARG;
      if (!part_ok(C[s], ldc[s], e - beg)) return GDN_ERR_INVALID_ARG;
      out.c[s] = C[s];
      out.ld[s] = ldc[s];
      out.vec[s] = ldc[s] % 8 == 0;
    } else {
      out.c[s] = out.c[n_parts - 1];
      out.ld[s] = out.ld[n_parts - 1];
      out.vec[s] = out.vec[n_parts - 1];
    }
    out.end[s] = e;
    beg = e;
  }
  const GemmGates gt{g, beta, A_log, dt_bias, param_is_fp32 ? 1 : 0, gate_col, Hv};
  return gemm_launch(A, lda, B, ldb, out, M, N, K, gt, stream);
}

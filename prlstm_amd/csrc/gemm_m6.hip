// Middle-sized fp32 products on the 16-bit matrix cores: the layouts of gemm_x6.hip
// (C = A B^T + bias, A^T B, A B) for products too small or too ragged to fill the chip with
// its 256-row tiles -- input projections, weight gradients and dx of ordinary batches
// (_torch.py:96, :157-162, _parallel.py:56).  Same arithmetic: the exact three-way bf16 split
// (split_bf16.h), six piece products, fp32 accumulation.
//
// What bounds it: the six products of a k-step take 96 ns of matrix time per 32x32 tile where
// the fp32 instruction takes 240, but each tile has to fetch and split its own operands, and a
// middle-sized product gives each CU only a few tiles.  A slice of one workgroup per CU takes
// 1.3 us (0.35 of them products; timing variants without the split, the loads or the products
// each save only 5-25%), of two 1.9 us, so it is the chain load - split - LDS - barrier -
// fragments - products, not any one unit.  us, the fp32 kernel against this one:
//   700 x 2600 x 650 A B^T 54 / 35;       2000 x 2052 x 300 A B^T 53 / 30
//   2600 x 650 x 700 A^T B 59 / 36;       700 x 650 x 2600 A B 80 / 37
//   5000 x 4096 x 256 A B^T 208 / 89 and 2100 x 1050 x 8000 A^T B 850 / 281 (before: the
//   masked instances of gemm_x6.hip)
// Hence:
//  * 128 x 64 output tiles on 4 waves, 32-deep
//    k-slices in one LDS buffer of 46 KB, so that two or three workgroups share a CU and
//    cover each other's loads, splits and barriers (the large kernel's 147 KB tile has no
//    neighbour).  The next slice's loads are issued before a slice's products.
//  * Operands are read as raw buffers with 16-byte loads that need 4-byte alignment only;
//    rows past the matrix read 0 or other rows, and only reach elements of C that are not
//    stored.  So every shape, aligned or not, runs the one kernel; the slice that holds the
//    last k is read element by element where a 16-byte load would straddle the end.
//  * The accumulators restart every 64 k and are added into a second fp32 sum, over at most
//    kSplitLongKRun k for A^T B and A B (A B^T: where a workspace is given and fewer than 256
//    tiles are there to run); splits are added in fp64.
//    (Without it the error of A B^T grew past the fp32 kernel's, which split K over waves.)
//
// Non-finite operands: a piece product of an infinite value is NaN wherever the other
// operand's piece is 0, so a tile whose result holds a NaN is computed again with the fp32
// instruction, which gives the IEEE result (the same for values beyond the bf16 range).
#include <algorithm>

#include "gemm_core.h"
#include "split_bf16.h"

namespace hsl {
namespace {

constexpr int kMBM = 128, kMBN = 64, kMBK = 32;
constexpr int kMLD = kMBK + 8;  // LDS row stride in bf16 elements (80 bytes: conflict-free 128-bit reads)
constexpr int kMThreads = 256;
constexpr int kMFold = 2;       // slices (64 k) per fold

struct M6Args {
  const float* A;
  const float* B;
  const float* bias;  // [N] or null (direct output only)
  float* out;         // C (ldc), or split-K planes [split][M][N]
  int M, N, K, lda, ldb, ldc;
  int kps;  // k per split, a multiple of kMBK
  int partial;
  int tiles_m, tiles_n;
};

// One operand's share of a ROWS x 32-k slice, L 16-byte loads per thread.
//  KC (k contiguous, [row][k]): load j of thread t is row c / 8, k-quad c % 8 (c = t + 256 j).
//  !KC ([k][row]): thread t loads rows 4 (t / 16) .. +3 (+ 64 s) at k-rows 2 (t % 16) and + 1
//      and writes each row's k-pair as one 32-bit word per piece.
template <bool KC, int ROWS>
struct M6Operand {
  static constexpr int L = ROWS / 32;
  static constexpr int P = ROWS * kMLD;  // elements of one piece
  __amdgpu_buffer_rsrc_t rs;
  unsigned off[L];  // byte offset of each load (advanced per slice)
  unsigned step;
  int k0[L];        // k of each load's first element, relative to the slice
  f4 v[L];
  __device__ __forceinline__ void init(const float* base, int ld, int r0, int rows, int K, int kbeg) {
    const size_t n = KC ? (size_t)(rows - 1) * ld + K : (size_t)(K - 1) * ld + rows;
    rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0, (int)(4 * n), 0x00020000);
    const int t = threadIdx.x;
    step = KC ? 4u * kMBK : 4u * kMBK * ld;
#pragma unroll
    for (int j = 0; j < L; ++j) {
      if constexpr (KC) {
        const int c = t + kMThreads * j;
        k0[j] = 4 * (c % 8);
        off[j] = 4u * ((unsigned)(r0 + c / 8) * ld + kbeg + k0[j]);
      } else {
        k0[j] = 2 * (t % 16) + (j & 1);
        off[j] = 4u * ((unsigned)(kbeg + k0[j]) * ld + r0 + 4 * (t / 16) + 64 * (j >> 1));
      }
    }
  }
  // elem: the slice holds the last k and 16-byte loads could straddle the buffer's end
  __device__ __forceinline__ void load(bool elem) {
#pragma unroll
    for (int j = 0; j < L; ++j) {
      if (!elem) {
        const u32x4 x = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off[j], 0, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) v[j][e] = __uint_as_float(x[e]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[j][e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, (int)(off[j] + 4u * e), 0, 0));
      }
      off[j] += step;
    }
  }
  // k >= left (k left in the matrix) of the slice in v set to 0 (k-contiguous operands; the
  // rows past K of the others lie past the buffer's end)
  __device__ __forceinline__ void mask(int left) {
    if constexpr (KC) {
#pragma unroll
      for (int j = 0; j < L; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[j][e] = k0[j] + e < left ? v[j][e] : 0.f;
    }
  }
  __device__ __forceinline__ void store(unsigned short* p0) const {
    const int t = threadIdx.x;
    if constexpr (KC) {
#pragma unroll
      for (int j = 0; j < L; ++j) {
        const int c = t + kMThreads * j;
        unsigned lo[3], hi[3];
        split2(v[j][0], v[j][1], lo);
        split2(v[j][2], v[j][3], hi);
#pragma unroll
        for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x2*>(p0 + q * P + (c / 8) * kMLD + 4 * (c % 8)) = u32x2{lo[q], hi[q]};
      }
    } else {
#pragma unroll
      for (int s = 0; s < L / 2; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          unsigned pc[3];
          split2(v[2 * s][i], v[2 * s + 1][i], pc);
#pragma unroll
          for (int q = 0; q < 3; ++q)
            *reinterpret_cast<unsigned*>(p0 + q * P + (4 * (t / 16) + 64 * s + i) * kMLD + 2 * (t % 16)) = pc[q];
        }
    }
  }
};

// element (row, k) of an operand; anything outside reads 0
template <bool KC>
__device__ __forceinline__ float m6_at(const float* p, int ld, int row, int k, int rows, int kend) {
  return row < rows && k < kend ? p[KC ? (size_t)row * ld + k : (size_t)k * ld + row] : 0.f;
}

template <bool AKC, bool BKC>
__global__ __launch_bounds__(kMThreads, 3) void gemm_m6_kernel(M6Args g) {
  constexpr int BN = kMBN, WM = 2, TM = kMBM / WM, FM = TM / 32;  // waves 2 x 2, one 32-column fragment each
  using OpA = M6Operand<AKC, kMBM>;
  using OpB = M6Operand<BKC, BN>;
  __shared__ __attribute__((aligned(16))) unsigned short sm[3 * (OpA::P + OpB::P)];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const int half = lane >> 5, r32 = lane & 31;
  int tm, tn;
  gemm_tile_order(g.tiles_m, g.tiles_n, &tm, &tn);
  const int m0 = tm * kMBM, n0 = tn * BN;
  const int kbeg = blockIdx.z * g.kps, kend = min(g.K, kbeg + g.kps);
  const int nk = (kend - kbeg + kMBK - 1) / kMBK;
  OpA oa;
  OpB ob;
  oa.init(g.A, g.lda, m0, g.M, g.K, kbeg);
  ob.init(g.B, g.ldb, n0, g.N, g.K, kbeg);
  const bool holds_end = kend == g.K;
  const bool elem_a = holds_end && (AKC ? g.K : g.M) % 4 != 0, elem_b = holds_end && (BKC ? g.K : g.N) % 4 != 0;

  f16v acc[FM];
  f16v tot[FM];
#pragma unroll
  for (int i = 0; i < FM; ++i) acc[i] = tot[i] = f16v{};
  auto fold = [&]() {
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      tot[i] += acc[i];
      acc[i] = f16v{};
    }
  };
  const unsigned short* const fa0 = sm + (wm * TM + r32) * kMLD + 8 * half;
  const unsigned short* const fb0 = sm + 3 * OpA::P + (wn * 32 + r32) * kMLD + 8 * half;
  oa.load(nk == 1 && elem_a);
  ob.load(nk == 1 && elem_b);
  for (int s = 0; s < nk; ++s) {
    if (s + 1 == nk && kend - kbeg < nk * kMBK) {  // the last slice ends inside
      oa.mask(kend - kbeg - s * kMBK);
      ob.mask(kend - kbeg - s * kMBK);
    }
    if (s > 0) lds_barrier();  // the previous slice has been read
    oa.store(sm);
    ob.store(sm + 3 * OpA::P);
    if (s + 1 < nk) {
      oa.load(s + 2 == nk && elem_a);
      ob.load(s + 2 == nk && elem_b);
    }
    lds_barrier();
#pragma unroll
    for (int ks = 0; ks < kMBK / 16; ++ks) {
      u32x4 fa[3][FM], fb[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        fb[q] = *reinterpret_cast<const u32x4*>(fb0 + q * OpB::P + 16 * ks);
#pragma unroll
        for (int i = 0; i < FM; ++i)
          fa[q][i] = *reinterpret_cast<const u32x4*>(fa0 + q * OpA::P + 32 * i * kMLD + 16 * ks);
      }
#pragma unroll
      for (int pp = 0; pp < 6; ++pp)
#pragma unroll
        for (int i = 0; i < FM; ++i) acc[i] = mfma_bf16(fa[kPa[pp]][i], fb[kPb[pp]], acc[i]);
    }
    if ((s + 1) % kMFold == 0 || s + 1 == nk) fold();
  }

  bool nan = false;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) nan = nan || tot[i][r] != tot[i][r];
  if (__any(nan)) {  // non-finite operands: this wave's part again on the fp32 instruction
#pragma unroll
    for (int i = 0; i < FM; ++i) tot[i] = f16v{};
    for (int k = kbeg; k < kend; k += 2) {
      const float b = m6_at<BKC>(g.B, g.ldb, n0 + wn * 32 + r32, k + half, g.N, kend);
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const float a = m6_at<AKC>(g.A, g.lda, m0 + wm * TM + 32 * i + r32, k + half, g.M, kend);
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[i], 0, 0, 0);
      }
      if ((k + 2 - kbeg) % (kMFold * kMBK) == 0) fold();
    }
    fold();
  }

  float* const out = g.partial ? g.out + (size_t)blockIdx.z * g.M * g.N : g.out;
  const int ldo = g.partial ? g.N : g.ldc;
  const int n = n0 + wn * 32 + r32;
  if (n >= g.N) return;
  const float bv = !g.partial && g.bias ? g.bias[n] : 0.f;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = m0 + wm * TM + 32 * i + 8 * (r >> 2) + 4 * half + (r & 3);
      if (m < g.M) out[(size_t)m * ldo + n] = tot[i][r] + bv;
    }
}

template <bool AKC, bool BKC>
void m6_launch(M6Args& g, int splits, hipStream_t s) {
  g.tiles_m = (g.M + kMBM - 1) / kMBM;
  g.tiles_n = (g.N + kMBN - 1) / kMBN;
  hipLaunchKernelGGL((gemm_m6_kernel<AKC, BKC>), dim3(g.tiles_m * g.tiles_n, 1, splits), dim3(kMThreads), 0,
                     s, g);
}

}  // namespace

int gemm_m6_splits(int M, int N, int K, int trans_a, int trans_b, int lda, int ldb) {
  // Fewer than 64 columns stay on the fp32 kernel's 32 x 32 tiles, whose four waves cut K: a 128 x
  // 64 tile would be half padding and wait out K alone (A B^T 1000 x 60 x 300 7 us, here 18; 256 x 33
  // x 4096 51, 167; the parallel backward at T148 B3 D60 H122 45, 71), and its fp64-folded sums of
  // 32 k are nearer to 64 bits (dW_ih 512 x 40 x 512 7.2e-8, here 1.46e-7), also where this kernel
  // is the faster one (M K above 6e6: the backward at T4000 B4 D40 H1024 450 us, here 318)
  if ((trans_a && trans_b) || M < 64 || N < 64 || K < 64) return 0;
  // a handful of tiles is all latency: ragged products of 1e6 to 6e6 multiply-adds take 0.7 to 0.9
  // of the fp32 kernel's 12 to 29 us here, those of 3e5 twice its 4 (whole ones: see stays_fp32 in
  // gemm.hip).  The line is above where the gain begins.
  if ((double)M * N * K < 6e6) return 0;
  // operands are addressed as raw buffers with 32-bit offsets (a tile's rows may start past the end)
  const size_t a = (size_t)((trans_a ? K : M) + 256) * lda, b = (size_t)((trans_b ? N : K) + 256) * ldb;
  if (a >= ((size_t)1 << 29) || b >= ((size_t)1 << 29)) return 0;
  const long tiles = (long)((M + kMBM - 1) / kMBM) * ((N + kMBN - 1) / kMBN);
  // A B^T, without the depth bound, is not split once each CU has a workgroup: its planes cost
  // more than its depth (2100 x 2048 x 512 in one split 43 us, in two 53; 700 x 2600 x 650 36, 34)
  if (!trans_a && trans_b && tiles >= 256) return 1;
  long s = (768 + tiles - 1) / tiles;  // three workgroups per CU
  s = std::min(s, (long)K / 256);
  s = std::max(s, (long)(K + kSplitLongKRun - 1) / kSplitLongKRun);
  return (int)std::max(1L, std::min(s, 64L));
}

int gemm_m6_run(const float* A, const float* B, const float* bias, float* C, float* partial, int M, int N, int K,
                int lda, int ldb, int ldc, int trans_a, int trans_b, int splits, hipStream_t s, int* used) {
  if (splits < 1 || (splits > 1 && !partial)) splits = 1;
  M6Args g{A, B, partial ? nullptr : bias, partial ? partial : C, M, N, K, lda, ldb, ldc, 0, partial ? 1 : 0, 0, 0};
  g.kps = ((K + splits - 1) / splits + kMBK - 1) / kMBK * kMBK;
  const int n = (K + g.kps - 1) / g.kps;
  if (used) *used = n;
  if (!trans_a && trans_b)
    m6_launch<true, true>(g, n, s);
  else if (trans_a)
    m6_launch<false, false>(g, n, s);
  else
    m6_launch<true, false>(g, n, s);
  HSL_HIP(hipGetLastError());
  return HSL_OK;
}

}  // namespace hsl

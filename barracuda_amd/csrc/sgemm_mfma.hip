// sgemm_mfma.hip -- f32 GEMM on the gfx950 matrix cores.
//
// Replaces MatMul::execute (crates/barracuda/src/ops/matmul.rs:89-214; WGSL
// kernels K1 shaders/math/matmul_gpu_evolved_f64.wgsl, K2
// matmul_cpu_tiled_f64.wgsl, K3 matmul_tiled_f64.wgsl), MatmulTiled
// (ops/matmul_tiled.rs:62-122) and BatchMatMul (ops/batch_matmul.rs:47-144,
// K5 batch_matmul_f64.wgsl).  Contract: C[m,n] = sum_p A[m,p] B[p,n], f32
// inputs, f32 accumulation, row-major.
//
// Design:
//   * Each f32 is split exactly into three bf16 parts on its way into LDS and a product is six
//     bf16 part products accumulated in f32 (bch_internal.h, split8): 16 k of a 32 x 32 block are
//     six v_mfma_f32_32x32x16_bf16 (192 matrix-core cycles) instead of eight
//     v_mfma_f32_32x32x2_f32 (512).  Error against 64 bits (2-norm, N(0,1) inputs, f32 -> split):
//     4096^3 1.1e-6 -> 1.0e-6, 1024^3 5.7e-7 -> 4.9e-7, 256^3 2.9e-7 -> 2.3e-7 (fewer roundings of
//     the accumulator per k).  Blocks whose operands the parts cannot stand for are redone on
//     the f32 instruction (end of the kernel).  Same box, against f32 MFMAs (us): 4096^3 934 -> 578
//     (147 -> 238 TFLOP/s), 16 x 1024^3 247 -> 159, 2047 x 3001 x 1537 284 -> 110, 512 x 11008 x
//     4096 and back with bias and GELU 717 -> 500.
//   * What bounds it: with a workgroup on every CU the clock.  64 workgroups of 256 x 256 run
//     at 80% of the matrix-core peak (3.2 us per 32 k), 256 of them at 57% (4.5 us).  Splitting
//     once per workgroup on the way into LDS, not once per fragment, keeps the conversions (5.5
//     VALU operations per element) at a sixth of the issue slots.
//   * Operand layout of the 32x32x16 instruction: lane l holds row l % 32 of A (column of B), k
//     8 (l / 32) .. + 7; result value r of lane l is C[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].
//     LDS keeps each part as [k octet][row][8 k]: a fragment is one 128-bit read of 32
//     consecutive rows, free of bank conflicts, and B given as [k][n] is transposed by the
//     conversion itself, which packs pairs along k.
//   * LDS is double-buffered, one barrier per pass, the next pass's first fragments read across
//     it (see the loop); one register set stages the global loads.
//   * Workgroup -> tile mapping is XCD-aware: gfx950 dispatches workgroups
//     round-robin over 8 XCDs, so consecutive workgroup ids are remapped to
//     one XCD's contiguous range of tiles, then walked in groups of 8 tile
//     rows so concurrently running tiles share A and B panels in that
//     XCD's L2.  A batched launch gives each XCD a contiguous run of
//     (batch, tile) slots, i.e. whole batches where they divide the run.
//   * CHECK=false needs m % BM == 0, n % BN == 0, k % BK == 0, lda/ldb/
//     strides multiples of 4 and 16-byte aligned A/B; CHECK=true handles any shape and alignment:
//     rows and columns outside the matrix are read from its last ones and not stored, and only
//     the pass with the k remainder, taken first, loads element by element.
//   * TB: B is given as [n][k] (ldb >= k), C = A B^T -- the linear layer's
//     y = x W^T with W [out, in] (shaders/misc/linear_f64.wgsl, the layers of
//     nn/fused_mlp.rs:38-168); it is loaded like A.
//   * Epilogue: C = act(acc (+ bias[col])) with act none, ReLU or GELU (tanh
//     form), fused into the store -- linear_f64.wgsl adds the bias after the
//     dot product, and fused_mlp runs relu_f64.wgsl (gelu_f64.wgsl for a GELU
//     layer) as a separate pass over the output.
#include "bch_internal.h"

#include <stdint.h>

#include <algorithm>
#include <string>
#include <type_traits>

namespace {

using bch::bf16_mm;
using bch::f32x16;
using bch::split8;
using bch::u32x4;

// Workgroup shapes.  BM x BN x BK name the tile; KS is the k-depth of one LDS buffer (a pass of
// the loop), WM x WN the wavefront grid.  Two wavefronts per SIMD everywhere but on the small
// tile: one's conversions and LDS reads run under the other's MFMAs.  Measured on one box
// (TFLOP/s, the first number four wavefronts with KS 16): 256 x 128 at 2048 x 4096 x 2048 166 ->
// 209 (4 x 2, KS 32), 128 x 128 at 2048^3 156 -> 189 (2 x 4, KS 32).
template <int BM, int BN>
struct Shape {};
template <>
struct Shape<256, 256> { static constexpr int WM = 2, WN = 4, KG = 1, KS = 16; };
template <>
struct Shape<256, 128> { static constexpr int WM = 4, WN = 2, KG = 1, KS = 32; };
template <>
struct Shape<128, 128> { static constexpr int WM = 2, WN = 4, KG = 1, KS = 32; };
template <>
struct Shape<64, 64> { static constexpr int WM = 2, WN = 2, KG = 2, KS = 64; };

template <int BM, int BN, int BK>
struct Cfg {
  using S = Shape<BM, BN>;
  static constexpr int KS = S::KS, WM = S::WM, WN = S::WN, KG = S::KG;
  static constexpr int NT = 64 * WM * WN * KG;              // threads per workgroup
  static constexpr int NO = KS / 8;                         // 8-wide k octets per pass
  static constexpr int PAD = 128 / NO;                      // bytes between octets (see the kernel)
  static constexpr int ASTR = BM * 16 + PAD, BSTR = BN * 16 + PAD;  // bytes of one octet of one part
  static constexpr int ABYTES = 3 * NO * ASTR, BUF = ABYTES + 3 * NO * BSTR;
  static constexpr int LDS_BYTES = 2 * BUF;
  static constexpr int CA = BM * NO / NT, CB = BN * NO / NT;  // octets of A and of B per thread
  static constexpr int TM = BM / WM / 32, TN = BN / WN / 32;  // MFMA blocks per wavefront
  static_assert(CA * NT == BM * NO && CB * NT == BN * NO, "tile must split evenly over the threads");
  static_assert(BK % KS == 0, "a k-tile is whole passes");
  static_assert(BN % 64 == 0, "a wavefront's columns of a [k][n] B share one octet");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS");
};

// Eight consecutive floats; only 4-byte aligned unless ALIGNED.
template <bool ALIGNED>
__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
  typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
  using V = std::conditional_t<ALIGNED, bch::f32x4, f32x4u>;
  const V x = *reinterpret_cast<const V*>(p), y = *reinterpret_cast<const V*>(p + 4);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = x[e];
    v[4 + e] = y[e];
  }
}

// ---- where the parts cannot stand for the floats: again on v_mfma_f32_32x32x2_f32 ----
// Operands that are infinite, NaN or 2^111 and more, and sums from 2^96, leave values that are not
// finite.  Whether any of a wavefront's NB blocks holds one; if so want[b / TN] gets bit 16 (b % TN)
// + r for each such value r of block b.
template <int NB, int TN>
__device__ __forceinline__ bool non_finite(const f32x16* x, unsigned* want) {
  static_assert(16 * TN <= 32, "a bit a value");
  float z = 0.0f;
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) z = fmaf(x[b][r], 0.0f, z);
#pragma unroll
  for (int i = 0; i < NB / TN; ++i) want[i] = 0;
  if (!__any(z != 0.0f)) return false;
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      want[b / TN] |= __builtin_isfinite(x[b][r]) ? 0u : 1u << (16 * (b % TN) + r);
  return true;
}

// sum: the product of this lane's row at qa and its columns at qb, TN blocks of a block row, by one
// wavefront straight from global memory.  Chunk c of nc is the 16 k from kof(c), then come the k
// from kr to K: lane half lh loads 8 consecutive k of its row and columns and step e contracts k e
// and 8 + e; two chunks are in flight.  Ends once every wanted value is NaN, which no further k
// changes.  A wavefront reads its panels alone, 10 bytes of L2 traffic per 100 FLOP: a few block
// rows cost their latency, a whole matrix twice the f32 instruction's time.  Measured (us, one
// box; a kernel on that instruction throughout / a k pair loaded, then multiplied, at a time /
// this): 4096^3 with one NaN in A 938 / 3230 / 736, with a row of NaN in B at half of k 997 / 3170 /
// 1553, with every sum past 2^96 936 / 3410 / 2390; 1024^3 with one NaN 27 / 105 / 38; 512 x 4096 x
// 11008 with one NaN 382 / 1140 / 251.  Fewer k than a pass: 4096 x 4096 x 8 22 / 17 / 19, x 31
// 29 / 19 / 19, 512 x 512 x 8 7.1 / 6.2 / 7.9, x 31 9.4 / 9.9 / 10.1.
template <int TN, bool TB, class KOf>
__device__ __forceinline__ void redo_f32(unsigned want, int nc, KOf&& kof, int kr, int K, int lh, const float* qa,
                                         const float* const (&qb)[TN], int ldb, f32x16 (&sum)[TN]) {
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) sum[j][r] = 0.0f;
  float a[2][8], b[2][TN][8];
  auto load = [&](int s, int c) {
    const int k0 = kof(min(c, nc - 1)) + 8 * lh;
    load8<false>(qa + k0, a[s]);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if constexpr (TB) {
        load8<false>(qb[j] + k0, b[s][j]);
      } else {
        const float* p = qb[j] + (long long)k0 * ldb;
#pragma unroll
        for (int e = 0; e < 8; ++e, p += ldb) b[s][j][e] = *p;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto step = [&](int s, int e) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
      sum[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s][e], b[s][j][e], sum[j], 0, 0, 0);
  };
  auto multiply = [&](int s) {
#pragma unroll
    for (int e = 0; e < 8; ++e) step(s, e);
    __builtin_amdgcn_sched_barrier(0);
  };
  if (nc > 0) load(0, 0);
#pragma unroll 1
  for (int c = 0; c < nc; c += 2) {
    load(1, c + 1);
    multiply(0);
    load(0, c + 2);
    if (c + 1 < nc) multiply(1);
    unsigned nan = 0;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) nan |= sum[j][r] != sum[j][r] ? 1u << (16 * j + r) : 0u;
    if (!__any((want & ~nan) != 0)) return;
  }
#pragma unroll 1
  for (int kb = kr; kb < K; kb += 16) {  // step e: k 2 e and 2 e + 1, zeros from K on
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (kb + 2 * e < K) {
        const int k = kb + 2 * e + lh, kc = min(k, K - 1);
        const float x = qa[kc];
        a[0][e] = k < K ? x : 0.0f;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const float y = TB ? qb[j][kc] : qb[j][(long long)kc * ldb];
          b[0][j][e] = k < K ? y : 0.0f;
        }
      }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (kb + 2 * e < K) step(0, e);
  }
}

// CHECK: any sizes (rows and columns outside the matrix are read from its last ones and not
// stored; a k remainder is taken by the first pass).  V4: 16-byte aligned rows.
template <int BM, int BN, int BK, bool CHECK, bool TB, bool EPI, bool V4 = false, bool HY = false>
__global__ __launch_bounds__((Cfg<BM, BN, BK>::NT)) void sgemm_mfma_kernel(
    int M, int N, int K, const float* __restrict__ A, int lda, long long sA,
    const float* __restrict__ B, int ldb, long long sB, float* __restrict__ C,
    int ldc, long long sC, int tiles_m, int tiles_n, const float* __restrict__ bias, int act,
    int hy_ndp, int hy_r, int hy_kt, float* __restrict__ hy_P, long long sAz, long long sBz, long long sCz) {
  using G = Cfg<BM, BN, BK>;
  constexpr int KS = G::KS, NO = G::NO, TM = G::TM, TN = G::TN;
  extern __shared__ float4 smem4[];
  char* const smem = reinterpret_cast<char*>(smem4);

  // ---- tile mapping (XCD-aware, grouped) ----
  const int ntiles = tiles_m * tiles_n;
  int p = blockIdx.x;
  long long bz = blockIdx.y;
  bool by_xcd = false;  // batches: (batch, tile) slots remapped XCD-contiguously
  if constexpr (!HY && !CHECK) {
    // Workgroups are dispatched round-robin over the 8 XCDs in linear id order (x fastest), so
    // a batch's tiles were spread over all eight L2s.  Each XCD takes a contiguous run of the
    // (batch, tile) slots instead: whole batches where a batch's tiles divide the run, each
    // batch's A and B then read into one L2.  Same box, three runs each (us): 16 x 1024^3 158.7 ->
    // 154.5, 8 x 1024^3 87.1 -> 84.8, 24 x 1024^3 263.7 -> 255.4, 64 x 512^3 86.6 -> 83.0, 32 x 1024
    // x 1024 x 512 165.7 -> 160.5, 4 x 2048 x 2048 x 1024 154.0 -> 153.0, 16 x 1024 x 1024 x 4096 640
    // -> 601.  The guarded tiles and split-K grids (slices in z) keep the dispatch order, which
    // their plans were measured in; remapped, batches of them would gain 1 to 5% (24 x 1000 x 1000
    // x 2000 524 -> 499, 8 x 256 x 512 x 4096 57.5 -> 54.7), single matrices nothing.
    const long long slots = (long long)gridDim.x * gridDim.y;
    if (gridDim.y > 1 && gridDim.z == 1 && (slots & 7) == 0) {
      const long long L = (long long)blockIdx.y * gridDim.x + blockIdx.x;
      const long long q = (L & 7) * (slots >> 3) + (L >> 3);
      bz = q / gridDim.x;
      p = (int)(q - bz * gridDim.x);
      by_xcd = true;
    }
  }
  int lt = p;
  bool tail = false;  // HY: this workgroup computes one k-slice of one of the last hy_r tiles
  int hy_slot = 0, hy_slice = 0;
  if constexpr (!HY) {
    if ((ntiles & 7) == 0 && !by_xcd) lt = (p & 7) * (ntiles >> 3) + (p >> 3);
  } else {
    // whole tiles 0 .. hy_ndp - 1 first (hy_ndp fills whole rounds), XCD-contiguous; then
    // the k-slices of tiles hy_ndp .. hy_ndp + hy_r - 1, slice-major and XCD-contiguous,
    // so that an XCD's workgroups run neighbouring tiles over the same k range
    if (p < hy_ndp) {
      if ((hy_ndp & 7) == 0) lt = (p & 7) * (hy_ndp >> 3) + (p >> 3);
    } else {
      const int nt = (int)gridDim.x - hy_ndp;
      int q = p - hy_ndp;
      if ((nt & 7) == 0) q = (q & 7) * (nt >> 3) + (q >> 3);
      hy_slice = q / hy_r;
      hy_slot = q - hy_slice * hy_r;
      lt = hy_ndp + hy_slot;
      tail = true;
    }
  }
  constexpr int GROUP = 8;
  const int group_size = GROUP * tiles_n;
  const int g = lt / group_size;
  const int first_m = g * GROUP;
  const int gm = min(tiles_m - first_m, GROUP);
  const int within = lt - g * group_size;
  const int tile_m = first_m + within % gm;
  const int tile_n = within / gm;
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  A += bz * sA;
  B += bz * sB;
  C += bz * sC;
  if (gridDim.z > 1) {  // split over k: blockIdx.z is the slice (its A, B offset and partial), hy_kt deep
    const long long zz = blockIdx.z;
    A += zz * sAz;
    B += zz * sBz;
    C += zz * sCz;
    K = min(hy_kt, K - (int)zz * hy_kt);
  }
  if constexpr (HY) {
    if (tail) {  // k-tiles hy_slice * hy_kt .. + hy_kt - 1, as a product of K = hy_kt * BK
      const long long k0 = (long long)hy_slice * hy_kt * BK;
      A += k0;
      B += TB ? k0 : k0 * ldb;
      K = hy_kt * BK;
    }
  }

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, lh = lane >> 5;
  const int kg = G::KG > 1 ? wave / (G::WM * G::WN) : 0;  // this wavefront's share of a pass's k
  const int wm = (wave / G::WN % G::WM) * (BM / G::WM);
  const int wn = (wave % G::WN) * (BN / G::WN);

  // ---- global -> registers: octets of 8 k of one row of A (column of B) ----
  // A row-major operand (A, and B given as [n][k]): octet ch covers row ch / NO, k 8 (ch % NO) ..
  // +7 of the pass, two 128-bit loads.  A [k][n] B: octet ch covers column ch % BN, k 8 (ch / BN)
  // .. +7, eight 32-bit loads of 64 consecutive columns by a wavefront, its row offsets scalar;
  // packing pairs along k in the conversion is the transpose.
  constexpr bool AL = !CHECK || V4;
  float ra[G::CA][8], rb[G::CB][8];
  const float* pa[G::CA];
  const float* pb[G::CB];
#pragma unroll
  for (int c = 0; c < G::CA; ++c) {
    const int ch = tid + c * G::NT;
    const int r = CHECK ? min(m0 + ch / NO, M - 1) : m0 + ch / NO;
    pa[c] = A + (long long)r * lda + 8 * (ch % NO);
  }
#pragma unroll
  for (int c = 0; c < G::CB; ++c) {
    const int ch = tid + c * G::NT;
    if constexpr (TB) {
      const int r = CHECK ? min(n0 + ch / NO, N - 1) : n0 + ch / NO;
      pb[c] = B + (long long)r * ldb + 8 * (ch % NO);
    } else {
      const int oct = wave / (BN / 64) + c * (G::NT / BN);  // ch / BN, uniform over the wavefront
      pb[c] = B + (long long)(8 * oct) * ldb;
    }
  }
  // (TB unset) this thread's column of B; NT % BN == 0 or BN % NT == 0 keeps ch % BN simple
  int cb[G::CB];
#pragma unroll
  for (int c = 0; c < G::CB; ++c) {
    const int col = n0 + (tid + c * G::NT) % BN;
    cb[c] = CHECK ? min(col, N - 1) : col;
  }
  auto load_pass = [&](int k0) {
#pragma unroll
    for (int c = 0; c < G::CA; ++c) load8<AL>(pa[c] + k0, ra[c]);
#pragma unroll
    for (int c = 0; c < G::CB; ++c) {
      if constexpr (TB) {
        load8<AL>(pb[c] + k0, rb[c]);
      } else {
        const float* s = pb[c] + (long long)k0 * ldb;
#pragma unroll
        for (int e = 0; e < 8; ++e) rb[c][e] = s[(long long)e * ldb + (unsigned)cb[c]];
      }
    }
  };
  // the k remainder: k0 .. K - 1, zeros from K on (loads past K read the last k instead)
  auto load_rest = [&](int k0) {
#pragma unroll
    for (int c = 0; c < G::CA; ++c) {
      const int k = k0 + 8 * ((tid + c * G::NT) % NO);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = pa[c][min(k + e, K - 1) - k + k0];
        ra[c][e] = k + e < K ? v : 0.0f;
      }
    }
#pragma unroll
    for (int c = 0; c < G::CB; ++c) {
      const int k = k0 + 8 * (TB ? (tid + c * G::NT) % NO : wave / (BN / 64) + c * (G::NT / BN));
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int d = min(k + e, K - 1) - k + k0;
        const float v = TB ? pb[c][d] : pb[c][(long long)d * ldb + cb[c]];
        rb[c][e] = k + e < K ? v : 0.0f;
      }
    }
  };

  // ---- registers -> LDS: three bf16 parts per float ----
  // [buffer][A or B][part][octet][row][8 k]: a fragment read takes 16 bytes of 32 consecutive
  // rows, so it needs no padding; PAD shifts the octets so that the eight lanes of a store phase
  // (128 / NO bytes of each of NO octets of a row-major operand) cover different banks.
  auto store_a = [&](int buf) {
    char* s = smem + buf * G::BUF;
#pragma unroll
    for (int c = 0; c < G::CA; ++c) {
      const int ch = tid + c * G::NT;
      u32x4 q[3];
      split8(ra[c], q);
#pragma unroll
      for (int p3 = 0; p3 < 3; ++p3)
        *reinterpret_cast<u32x4*>(s + (p3 * NO + ch % NO) * G::ASTR + (ch / NO) * 16) = q[p3];
    }
  };
  auto store_b = [&](int buf) {
    char* s = smem + buf * G::BUF + G::ABYTES;
#pragma unroll
    for (int c = 0; c < G::CB; ++c) {
      const int ch = tid + c * G::NT;
      const int row = TB ? ch / NO : ch % BN, oct = TB ? ch % NO : ch / BN;
      u32x4 q[3];
      split8(rb[c], q);
#pragma unroll
      for (int p3 = 0; p3 < 3; ++p3) *reinterpret_cast<u32x4*>(s + (p3 * NO + oct) * G::BSTR + row * 16) = q[p3];
    }
  };

  // ---- LDS -> operand fragments: lane l takes row l % 32, k octet l / 32 ----
  constexpr int NS = KS / 16 / G::KG, NB = NS * TM;  // 16-k steps, block steps of a wavefront's pass
  const char* const a_base = smem + (2 * NS * kg + lh) * G::ASTR + (wm + li) * 16;
  const char* const b_base = smem + G::ABYTES + (2 * NS * kg + lh) * G::BSTR + (wn + li) * 16;
  auto read_a = [&](int buf, int kk, int i, u32x4 (&f)[3]) {
#pragma unroll
    for (int p3 = 0; p3 < 3; ++p3)
      f[p3] = *reinterpret_cast<const u32x4*>(a_base + buf * G::BUF + (p3 * NO + 2 * kk) * G::ASTR + i * 512);
  };
  auto read_b = [&](int buf, int kk, u32x4 (&f)[TN][3]) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int p3 = 0; p3 < 3; ++p3)
        f[j][p3] = *reinterpret_cast<const u32x4*>(b_base + buf * G::BUF + (p3 * NO + 2 * kk) * G::BSTR + j * 512);
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  // Pass t runs NB block steps (row block i of 16-k step kk); each reads the next step's
  // fragments first, so LDS latency hides under its 6 TN MFMAs.  Pass t + 1's octets are
  // converted and stored to the other buffer at the start of pass t, and pass t + 2's loads issue
  // right behind.  The barrier sits before the last step's MFMAs (fragments in registers): every
  // read of this buffer and every store of the next one is done, and the next pass's first reads
  // overlap those MFMAs.  The last pass reloads the last tile into the buffer no one reads again.
  // (A copy of the pass without them, for the end of the loop, spilled 256 VGPRs at 256 x 256.)
  u32x4 fa[2][3], fb[2][TN][3];
  const int nk = (K + KS - 1) / KS;
  const int rest = CHECK && K % KS != 0 ? 1 : 0;  // the remainder runs first, as pass 0
  auto pass = [&](auto par, int t) {
    constexpr int P = decltype(par)::value;  // pass parity: LDS buffer and fragment sets
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int kk = b / TM, i = b % TM;
      const int fs = (P * NB + b) & 1, bs = (P * NS + kk) & 1;
      constexpr int b1 = NB > 2 ? 1 : 0;
      if (b == 0) store_a(P ^ 1);
      if (b == b1) {
        store_b(P ^ 1);
        load_pass((min(t + 2, nk - 1) - rest) * KS);
      }
      if (b < NB - 1) {
        const int kn = (b + 1) / TM, in = (b + 1) % TM;
        read_a(P, kn, in, fa[fs ^ 1]);
        if (in == 0) read_b(P, kn, fb[bs ^ 1]);
      } else {
        __syncthreads();
        read_a(P ^ 1, 0, 0, fa[fs ^ 1]);
        read_b(P ^ 1, 0, fb[bs ^ 1]);
      }
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = bf16_mm(fa[fs][bch::kPartA[q]], fb[bs][j][bch::kPartB[q]], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Fewer k than one pass holds (K = 0 too): redo_f32 alone.
  const bool short_k = K < KS;
  if (!short_k) {
    if (rest)
      load_rest((nk - 1) * KS);
    else
      load_pass(0);
    store_a(0);
    store_b(0);
    load_pass((min(1, nk - 1) - (nk > 1 ? rest : 0)) * KS);
    __syncthreads();
    read_a(0, 0, 0, fa[0]);
    read_b(0, 0, fb[0]);
    int t = 0;
    for (; t + 1 < nk; t += 2) {
      pass(std::integral_constant<int, 0>{}, t);
      pass(std::integral_constant<int, 1>{}, t + 1);
    }
    if (t < nk) pass(std::integral_constant<int, 0>{}, t);
  }

  // ---- the k shares of a block added up, in share order ----
  if constexpr (G::KG > 1) {
    static_assert(G::KG == 2 && TM == 1 && TN == 1 && G::WM * G::WN * 4096 <= G::LDS_BYTES, "one block a wavefront");
    __syncthreads();  // the last pass's reads are done
    f32x16* const part = reinterpret_cast<f32x16*>(smem) + (wave % (G::WM * G::WN)) * 64 + lane;
    if (kg != 0) *part = acc[0][0];
    __syncthreads();
    if (kg != 0) return;
    acc[0][0] += *part;
  }

  // ---- scaled back; `want`: the values to compute again in f32 ----
  unsigned want[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] *= bch::kSplitUnscale;
  const bool redo = non_finite<TM * TN, TN>(&acc[0][0], want) || short_k;

  // ---- epilogue: value r of lane l is row 8*(r/4) + 4*lh + r%4, col li ----
  float* Pt = nullptr;
  if constexpr (HY) {
    if (tail) {  // the slice's sums, a whole BM x BN tile, into its slot of the partials
      Pt = hy_P + ((long long)hy_slice * hy_r + hy_slot) * (BM * BN);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            Pt[(wm + i * 32 + 8 * (r >> 2) + 4 * lh + (r & 3)) * BN + wn + j * 32 + li] = acc[i][j][r];
    }
  }
  const bool store = !short_k && !(HY && tail);
  if constexpr (!EPI) {
#pragma unroll
    for (int i = 0; i < TM && store; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int col = n0 + wn + j * 32 + li;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = m0 + wm + i * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
          if (!CHECK || (row < M && col < N)) C[(long long)row * ldc + col] = acc[i][j][r];
        }
        __builtin_amdgcn_sched_barrier(0);  // one block's addresses at a time: no spills
      }
    }
  } else if (store) {
    // bias and the activation are uniform over the launch (no divergence); one 32 x 32
    // block at a time, so only 16 accumulators are out of the AGPRs at once
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + wn + j * 32 + li;
      const float bj = bias ? (!CHECK || col < N ? bias[col] : 0.0f) : 0.0f;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = m0 + wm + i * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
          float v = acc[i][j][r] + bj;
          v = bch::activate(v, act);
          if (!CHECK || (row < M && col < N)) C[(long long)row * ldc + col] = v;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  if (!redo) return;

  // ---- the values that were not finite (all of a call with fewer k than a pass) again in f32 ----
  // After the stores and one block row at a time in a loop that is not unrolled: the accumulators'
  // registers are free, and the loop above keeps its own.
#pragma unroll 1
  for (int i = 0; i < TM; ++i) {
    unsigned w = 0;
#pragma unroll
    for (int ii = 0; ii < TM; ++ii) w = i == ii ? want[ii] : w;
    if (short_k) w = ~0u;
    if (!__any(w != 0)) continue;
    const float* qb[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = min(n0 + wn + j * 32 + li, N - 1);
      qb[j] = TB ? B + (long long)n * ldb : B + n;
    }
    f32x16 sum[TN];
    redo_f32<TN, TB>(w, K / 16, [](int c) { return 16 * c; }, K / 16 * 16, K, lh, A + (long long)min(m0 + wm + i * 32 + li, M - 1) * lda, qb, ldb, sum);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int lc = wn + j * 32 + li, col = n0 + lc;
      const float bj = EPI && bias && col < N ? bias[col] : 0.0f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int lr = wm + i * 32 + 8 * (r >> 2) + 4 * lh + (r & 3), row = m0 + lr;
        if (!(w >> (16 * j + r) & 1u)) continue;
        if (HY && tail)
          Pt[lr * BN + lc] = sum[j][r];
        else if (row < M && col < N)
          C[(long long)row * ldc + col] = EPI ? bch::activate(sum[j][r] + bj, act) : sum[j][r];
      }
    }
  }
}

template <int BM, int BN, int BK, bool CHECK, bool TB, bool EPI, bool V4 = false>
hipError_t launch_tiles(hipStream_t s, int batch, int m, int n, int k,
                        const float* A, int lda, long long sA, const float* B,
                        int ldb, long long sB, float* C, int ldc, long long sC,
                        const float* bias, int act, int nz = 1, int kc = 0, long long sAz = 0, long long sBz = 0,
                        long long sCz = 0) {
  using G = Cfg<BM, BN, BK>;
  const int tm = (m + BM - 1) / BM, tn = (n + BN - 1) / BN;
  const size_t lds = G::LDS_BYTES;
  auto kern = sgemm_mfma_kernel<BM, BN, BK, CHECK, TB, EPI, V4>;
  hipError_t e = bch::ensure_dynamic_lds(reinterpret_cast<const void*>(kern), (int)lds);
  if (e != hipSuccess) return e;
  if (batch > 65535 || nz > 65535) return hipErrorInvalidValue;
  hipLaunchKernelGGL(kern, dim3(tm * tn, batch, nz), dim3(G::NT), lds, s, m, n, k,
                     A, lda, sA, B, ldb, sB, C, ldc, sC, tm, tn, bias, act, 0, 0, kc, nullptr, sAz, sBz, sCz);
  return hipGetLastError();
}

// The hybrid launch (batch 1, K a multiple of BK): ndp whole tiles, then r tiles in
// S k-slices of kt k-tiles each into P (see HybPlan).
template <int BM, int BN, int BK, bool CHECK, bool TB, bool EPI, bool V4>
hipError_t launch_hyb_tiles(hipStream_t s, int m, int n, int k, const float* A, int lda, const float* B, int ldb,
                            float* C, int ldc, const float* bias, int act, int ndp, int r, int S, int kt, float* P) {
  using G = Cfg<BM, BN, BK>;
  const int tm = (m + BM - 1) / BM, tn = (n + BN - 1) / BN;
  const size_t lds = G::LDS_BYTES;
  auto kern = sgemm_mfma_kernel<BM, BN, BK, CHECK, TB, EPI, V4, true>;
  hipError_t e = bch::ensure_dynamic_lds(reinterpret_cast<const void*>(kern), (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3(ndp + r * S), dim3(G::NT), lds, s, m, n, k, A, lda, 0LL, B, ldb, 0LL, C, ldc,
                     0LL, tm, tn, bias, act, ndp, r, kt, P, 0LL, 0LL, 0LL);
  return hipGetLastError();
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

constexpr int kBK = 32;

// Tile choice: the tile with the least modelled time per 32 k of depth.  One workgroup of a tile
// alone on the chip takes `idle` us per 32 k, with one on every CU `full` us (the clock falls as
// more matrix cores run, and L2 is shared): measured at K 2048-4096 on one box, 256 x 256 3.2 /
// 4.5 (4096^3), 256 x 128 1.9 / 2.45, 128 x 128 1.1 / 1.42 (2048^3).  Whole rounds take `full`, a
// part-filled last one in between by its share of the CUs.  eff: the tiles' rates at whole
// rounds relative to 256 x 256, for the hybrid and mixed plans.
enum class Tile { k256x256, k256x128, k128x128 };

struct TileOpt { Tile t; int bm, bn; double eff, idle, full; };
constexpr TileOpt kTileOpts[] = {{Tile::k256x256, 256, 256, 1.0, 3.3, 4.65}, {Tile::k256x128, 256, 128, 0.966, 1.9, 2.45},
                                 {Tile::k128x128, 128, 128, 0.92, 1.08, 1.42}};
constexpr double kTileKtUs = 4.6;  // one 256 x 256 k-tile of 32 at whole rounds

// us per 32 k of `wgs` workgroups of tile o
double tile_kt_us(const TileOpt& o, long long wgs) {
  const long long cu = bch::device_cu_count();
  const long long r = wgs % cu;
  return (double)(wgs / cu) * o.full + (r ? o.idle + (o.full - o.idle) * (double)r / (double)cu : 0.0);
}

long long tile_count(const TileOpt& o, int batch, int m, int n) {
  return (long long)batch * ((m + o.bm - 1) / o.bm) * ((n + o.bn - 1) / o.bn);
}

Tile pick_tile(int batch, int m, int n) {
  Tile best = Tile::k256x256;
  double best_cost = 0.0;
  for (const TileOpt& o : kTileOpts) {
    const double cost = tile_kt_us(o, tile_count(o, batch, m, n));
    if (o.t == Tile::k256x256 || cost < best_cost * 0.999) {
      best = o.t;
      best_cost = cost;
    }
  }
  return best;
}

int tile_m(Tile t) { return t == Tile::k128x128 ? 128 : 256; }
int tile_n(Tile t) { return t == Tile::k256x256 ? 256 : 128; }

bool fast_ok(Tile t, int m, int n, int k, const float* A, int lda, long long sA, const float* B, int ldb,
             long long sB) {
  return m % tile_m(t) == 0 && n % tile_n(t) == 0 && k % kBK == 0 && lda % 4 == 0 && ldb % 4 == 0 &&
         sA % 4 == 0 && sB % 4 == 0 && aligned16(A) && aligned16(B);
}

// Guarded tiles with 16-byte loads of A's rows (and a [n][k] B's): bases, leading dimensions and
// batch strides that keep rows 16-byte aligned.  K and N multiples of 4 are the rule's own: the
// clamped loads would take any (a [k][n] B is loaded by columns, in any alignment), and the hybrid
// plan, which runs on aligned loads alone, with them.
bool vec4_ok(int n, int k, const float* A, int lda, long long sA, const float* B, int ldb, long long sB) {
  return k >= 4 && k % 4 == 0 && n % 4 == 0 && lda % 4 == 0 && ldb % 4 == 0 && sA % 4 == 0 && sB % 4 == 0 &&
         aligned16(A) && aligned16(B);
}

// k slices in grid.z (the split-K launch): slice z adds z * (sA, sB, sC) to the batch's operands
struct ZSplit {
  int nz = 1, kc = 0;  // slices, their depth (the last one takes what is left)
  long long sA = 0, sB = 0, sC = 0;
};

template <bool CHECK, bool TB, bool EPI, bool V4>
hipError_t launch_tile(Tile t, hipStream_t s, int batch, int m, int n, int k, const float* A, int lda,
                       long long sA, const float* B, int ldb, long long sB, float* C, int ldc, long long sC,
                       const float* bias, int act, const ZSplit& z) {
  switch (t) {
    case Tile::k256x256:
      return launch_tiles<256, 256, kBK, CHECK, TB, EPI, V4>(s, batch, m, n, k, A, lda, sA, B, ldb, sB, C, ldc, sC,
                                                             bias, act, z.nz, z.kc, z.sA, z.sB, z.sC);
    case Tile::k256x128:
      return launch_tiles<256, 128, kBK, CHECK, TB, EPI, V4>(s, batch, m, n, k, A, lda, sA, B, ldb, sB, C, ldc, sC,
                                                             bias, act, z.nz, z.kc, z.sA, z.sB, z.sC);
    default:
      return launch_tiles<128, 128, kBK, CHECK, TB, EPI, V4>(s, batch, m, n, k, A, lda, sA, B, ldb, sB, C, ldc, sC,
                                                             bias, act, z.nz, z.kc, z.sA, z.sB, z.sC);
  }
}

// mode 0: unguarded; 1: guarded, 16-byte aligned rows; 2: guarded, any alignment
template <bool TB, bool EPI>
hipError_t launch_tile_any(int mode, Tile t, hipStream_t s, int batch, int m, int n, int k, const float* A,
                           int lda, long long sA, const float* B, int ldb, long long sB, float* C, int ldc,
                           long long sC, const float* bias, int act, const ZSplit& z = ZSplit{}) {
  if (mode == 0)
    return launch_tile<false, TB, EPI, false>(t, s, batch, m, n, k, A, lda, sA, B, ldb, sB, C, ldc, sC, bias, act, z);
  if (mode == 1)
    return launch_tile<true, TB, EPI, true>(t, s, batch, m, n, k, A, lda, sA, B, ldb, sB, C, ldc, sC, bias, act, z);
  return launch_tile<true, TB, EPI, false>(t, s, batch, m, n, k, A, lda, sA, B, ldb, sB, C, ldc, sC, bias, act, z);
}

const char* tile_name(Tile t, int mode) {
  static const char* const names[3][3] = {
      {"sgemm_mfma_kernel<256,256,32,false>", "sgemm_mfma_kernel<256,256,32,true,v4>", "sgemm_mfma_kernel<256,256,32,true>"},
      {"sgemm_mfma_kernel<256,128,32,false>", "sgemm_mfma_kernel<256,128,32,true,v4>", "sgemm_mfma_kernel<256,128,32,true>"},
      {"sgemm_mfma_kernel<128,128,32,false>", "sgemm_mfma_kernel<128,128,32,true,v4>", "sgemm_mfma_kernel<128,128,32,true>"}};
  return names[static_cast<int>(t)][mode];
}

// ---- split-K for shapes whose tiles fill less than one round ----
// K is cut into S slices of whole k-tiles; the slices run as one launch of
// the tile kernel with the slice in grid.z (batch b, slice j: A + b sA + j kc,
// B + b sB + j kc rows -- or columns for B given as [n][k] -- into P[b][j],
// an m x n partial), then sgemm_splitk_reduce sums the S partials of each
// output in slice order (deterministic) and applies the epilogue.  Batches
// split the same way when all of their tiles together fill less than a
// round (4 x 512 x 512 x 4096: 64 tiles).  Tile and S are the modelled
// fastest: the rounds' time per 32 k (below) x k-tiles per slice, plus the
// partials' round trip ((2S + 1) M N floats at 5 TB/s), the reduce launch and
// each further round; a slice has at least kSplitMinKt k-tiles (the last one
// what is left, the remainder of K too), and the partials fit the cap.  The plan is made against
// a fixed cap, not the workspace at hand, so a shape always rounds the same
// way through bch_sgemm; bch_sgemm_noalloc plans against its 16 MiB scratch
// and can take fewer slices (within tolerance of bch_sgemm).  Measured (one
// box, us): 512 x 4096 x 11008 as 256 x 128 tiles in 4 slices 222 (128 x 128 in
// 2: 246, no split 381), 512 x 11008 x 4096 as 256 x 256 in 2 245 (256 x 128
// unsplit 262), 1024 x 1024 x 4096 as 128 x 128 in 4 60 (64 x 64 unsplit 76).
constexpr size_t kSplitWsMax = (size_t)256 << 20;
constexpr size_t kSplitWsSmall = bch::kSgemmFixedScratch;
constexpr int kSplitMinKt = 4;  // k-tiles per slice at least
constexpr double kTileFixedUs = 3.0;    // an unsplit launch's prologue and stores
constexpr double kSplitBytesUs = 5e6;   // the partials' round trip
constexpr double kSplitRoundUs = 1.5;   // a further round's prologue and stores
constexpr double kSplitFixedUs = 5.0;   // the reduce launch

struct SplitPlan {
  Tile t = Tile::k128x128;
  int S = 1;          // slices; 1: no split
  int kc = 0;         // their depth, a multiple of kBK
  double us = 0.0;    // modelled time
};

SplitPlan split_plan(int batch, int m, int n, int k, size_t cap = kSplitWsMax) {
  SplitPlan p;
  if (batch < 1 || k <= 0) return p;
  const long long cu = bch::device_cu_count();
  p.t = pick_tile(batch, m, n);
  const double mn = (double)batch * m * n * sizeof(float);
  const int nk = (k + kBK - 1) / kBK;
  // a part-filled round stays near `idle` up to half of the CUs (256 x 256: 64, 128 and 172
  // workgroups 3.2, 3.26 and 3.4 us per 32 k; 256 x 128: 1.85, 1.93 and 2.05)
  auto kt_us = [&](const TileOpt& o, long long wgs) {
    const double r = (double)(wgs % cu) / (double)cu;
    return (double)(wgs / cu) * o.full + (r > 0.0 ? o.idle + (o.full - o.idle) * r * r * r * r : 0.0);
  };
  for (const TileOpt& o : kTileOpts)
    if (o.t == p.t) {
      const long long tiles = tile_count(o, batch, m, n);
      if (tiles >= cu) return p;  // whole rounds: the data-parallel tiling or the hybrid plan
      p.us = nk * kt_us(o, tiles) + kTileFixedUs;
    }
  for (const TileOpt& o : kTileOpts) {
    const long long tiles = tile_count(o, batch, m, n);
    for (int kt = (nk + 1) / 2; kt >= kSplitMinKt; --kt) {  // k-tiles per slice
      const int sl = (nk + kt - 1) / kt;
      if (sl < 2 || (nk + sl - 1) / sl != kt) continue;  // the evenest cut into sl slices
      if ((size_t)sl * batch * m * n * sizeof(float) > cap) break;
      const long long rounds = (tiles * sl + cu - 1) / cu;
      const double us = kt * kt_us(o, tiles * sl) + kSplitRoundUs * (double)(rounds - 1) +
                        (2.0 * sl + 1.0) * mn / kSplitBytesUs + kSplitFixedUs;
      if (us < p.us) {
        p.t = o.t;
        p.S = sl;
        p.kc = kt * kBK;
        p.us = us;
      }
    }
  }
  return p;
}

int split_slices(int batch, int m, int n, int k, size_t cap = kSplitWsMax) {
  return split_plan(batch, m, n, k, cap).S;
}

// ---- small shapes: 64 x 64 x 64 tiles ----
// Where the planned tiles fill less than one round, 64 x 64 tiles put 4 to 16 times the
// workgroups on the CUs, with no k split, partials or reduce launch.  A pass is 64 k deep; the
// two halves of its k go to two sets of four wavefronts, whose sums meet in LDS at the end, so a
// SIMD always has a second wavefront to run while one converts, stores or waits.  Against four
// wavefronts and passes of 32 (same box, us): 256^3 8.3 -> 7.05, 512^3 13.7 -> 10.6, 1024^3 25.6 ->
// 20.6, 1024 x 1024 x 4096 95 -> 76.  (More loads in flight, 2 or 4 passes, changed nothing.)  A
// 64-k pass takes 1.0-1.2 us whatever the tile count up to a round.  Taken when the modelled time
// is under the split plan's; unguarded loads only (m, n, k multiples of 64, aligned operands).
constexpr int kSmallBK = 64;
constexpr double kSmallKtUs = 1.12;

bool small_tile_plan(int batch, int m, int n, int k) {
  if (batch < 1 || m % 64 != 0 || n % 64 != 0 || k <= 0 || k % kSmallBK != 0) return false;
  const SplitPlan p = split_plan(batch, m, n, k);
  if (p.us == 0.0) return false;  // whole rounds of the other tiles
  const long long cu = bch::device_cu_count();
  const long long t64 = (long long)batch * (m / 64) * (n / 64);
  return (double)((t64 + cu - 1) / cu) * (k / kSmallBK) * kSmallKtUs < p.us;
}

bool small_tile_ok(int batch, int m, int n, int k, const float* A, int lda, long long sA, const float* B, int ldb,
                   long long sB) {
  return small_tile_plan(batch, m, n, k) && lda % 4 == 0 && ldb % 4 == 0 && sA % 4 == 0 && sB % 4 == 0 &&
         aligned16(A) && aligned16(B);
}

// C[b][m][n] = act(sum over j < S of P[b][j][m][n] (+ bias[n])) for each of `batch` matrices
// (C[b] at C + b sC); V: four columns per thread (n % 4 == 0, ldc % 4 == 0, C 16-byte aligned)
template <bool V>
__global__ __launch_bounds__(256) void sgemm_splitk_reduce(int M, int N, int S, int batch, const float* __restrict__ P,
                                                           float* __restrict__ C, int ldc, long long sC,
                                                           const float* __restrict__ bias, int act) {
  const long long per = (long long)M * N;
  const int w = V ? 4 : 1;
  const long long total = per * batch / w;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    const long long ea = i * w;
    const long long b = ea / per, e = ea - b * per;
    const int m = (int)(e / N), n = (int)(e - (long long)m * N);
    const float* pb = P + b * S * per + e;
    float* cb = C + b * sC + (long long)m * ldc + n;
    if constexpr (V) {
      float4 acc = *reinterpret_cast<const float4*>(pb);
      for (int j = 1; j < S; ++j) {
        const float4 x = *reinterpret_cast<const float4*>(pb + j * per);
        acc.x += x.x;
        acc.y += x.y;
        acc.z += x.z;
        acc.w += x.w;
      }
      if (bias) {
        acc.x += bias[n];
        acc.y += bias[n + 1];
        acc.z += bias[n + 2];
        acc.w += bias[n + 3];
      }
      acc = make_float4(bch::activate(acc.x, act), bch::activate(acc.y, act), bch::activate(acc.z, act),
                        bch::activate(acc.w, act));
      *reinterpret_cast<float4*>(cb) = acc;
    } else {
      float acc = pb[0];
      for (int j = 1; j < S; ++j) acc += pb[j * per];
      if (bias) acc += bias[n];
      *cb = bch::activate(acc, act);
    }
  }
}

hipError_t launch_splitk_reduce(hipStream_t s, int m, int n, int S, int batch, const float* P, float* C, int ldc,
                                long long sC, const float* bias, int act) {
  const bool v = n % 4 == 0 && ldc % 4 == 0 && aligned16(C) && (batch == 1 || sC % 4 == 0) &&
                 (bias == nullptr || aligned16(bias));
  const long long work = (long long)m * n * batch / (v ? 4 : 1);
  const int blocks = (int)std::min<long long>((work + 255) / 256, 4096);
  if (v)
    hipLaunchKernelGGL(sgemm_splitk_reduce<true>, dim3(blocks), dim3(256), 0, s, m, n, S, batch, P, C, ldc, sC, bias,
                       act);
  else
    hipLaunchKernelGGL(sgemm_splitk_reduce<false>, dim3(blocks), dim3(256), 0, s, m, n, S, batch, P, C, ldc, sC, bias,
                       act);
  return hipGetLastError();
}

// ---- whole rounds data-parallel, the last round's tiles split over k (the hybrid plan) ----
// With T tiles on CU compute units, R = T / CU whole rounds and r = T mod CU
// tiles left over, the last round would run r workgroups of full length on
// r CUs.  Instead one launch runs the R * CU whole tiles and then the r tiles
// in S slices of equal k length (S * r <= CU), each slice's sums stored as a
// compact BM x BN tile; sgemm_tail_reduce adds each tile's S slices in slice
// order (deterministic) and applies the epilogue that the whole tiles apply
// in the kernel.  Every slice covers the same k-tiles of neighbouring tiles,
// so the slices of a round share A and B panels in L2 the way whole tiles do.
// The plan is modelled like the tile choice (k-tiles x tile area /
// efficiency per round; the partials' HBM traffic at 6.3 TB/s, one 256 x 256
// k-tile taking kTileKtUs) and used when it beats the best data-parallel tiling
// by 3%.  It needs K a multiple of 32 and unguarded or 16-byte aligned loads (vec4_ok);
// without the workspace (up to kHybWsMax) the data-parallel tiling runs.
constexpr size_t kHybWsMax = (size_t)256 << 20;
constexpr int kHybMinKt = 8;  // k-tiles per slice at least

struct HybPlan {
  Tile t = Tile::k256x256;
  int S = 0, ndp = 0, r = 0, kt = 0;  // slices, whole tiles, split tiles, k-tiles per slice
};

size_t hyb_bytes(const HybPlan& h) { return (size_t)h.S * h.r * tile_m(h.t) * tile_n(h.t) * sizeof(float); }

// cost_us (nullable): the modelled time of what the tile path then runs, the hybrid plan or the
// best data-parallel tiling
bool hyb_plan(int batch, int m, int n, int k, HybPlan& out, double* cost_us = nullptr) {
  if (batch != 1 || k <= 0 || k % kBK != 0 || split_slices(batch, m, n, k) > 1) return false;
  const long long cu = bch::device_cu_count();
  const int nk = k / kBK;
  double best_dp = 0.0, best = 0.0;
  bool found = false;
  for (const TileOpt& o : kTileOpts) {
    const long long T = (long long)((m + o.bm - 1) / o.bm) * ((n + o.bn - 1) / o.bn);
    const double per = o.bm * o.bn / 65536.0 / o.eff;  // one k-tile of this tile, in 256 x 256 k-tiles
    const double dp = (double)((T + cu - 1) / cu) * nk * per;
    if (best_dp == 0.0 || dp < best_dp) best_dp = dp;
    const long long R = T / cu, r = T % cu;
    if (R < 1 || r == 0) continue;
    int S = 0;
    for (int sl = 8; sl >= 2; --sl)
      if (sl * r <= cu && nk % sl == 0 && nk / sl >= kHybMinKt &&
          (size_t)sl * r * o.bm * o.bn * sizeof(float) <= kHybWsMax) {
        S = sl;
        break;
      }
    if (S == 0) continue;
    const double cost = (double)(R * nk + nk / S) * per + (2.0 * S + 1.0) * r * (o.bm * o.bn / 65536.0) * 0.009 + 0.45;
    if (!found || cost < best) {
      found = true;
      best = cost;
      out.t = o.t;
      out.S = S;
      out.ndp = (int)(R * cu);
      out.r = (int)r;
      out.kt = nk / S;
    }
  }
  const bool use = found && best < 0.97 * best_dp;
  if (cost_us) *cost_us = kTileKtUs * (use ? best : best_dp);
  return use;
}

// Modelled time (us) of a batch-1 call on the tile path: split-K, the hybrid plan or the best
// data-parallel tiling, whichever the tile path takes (given its workspace).
double tile_path_cost_us(int m, int n, int k) {
  double c = 0.0;
  const SplitPlan sp = split_plan(1, m, n, k);
  if (sp.S > 1) return sp.us;
  HybPlan h;
  if (k > 0 && k % kBK == 0) {
    hyb_plan(1, m, n, k, h, &c);
    return c;
  }
  // K not a multiple of the k-tile: data-parallel only
  const long long cu = bch::device_cu_count();
  double best = 0.0;
  for (const TileOpt& o : kTileOpts) {
    const long long T = (long long)((m + o.bm - 1) / o.bm) * ((n + o.bn - 1) / o.bn);
    const double t = (double)((T + cu - 1) / cu) * ((k + kBK - 1) / kBK) * kTileKtUs * o.bm * o.bn / 65536.0 / o.eff;
    if (best == 0.0 || t < best) best = t;
  }
  return best;
}

// ---- whole rounds of 256 x 256 tiles on part of C, the rest planned on its own (the mixed plan) ----
// The hybrid plan's split tiles and the smaller tiles it picks to fill the last round cost
// efficiency over the whole matrix.  Where the 256 x 256 tiles make at least one whole round,
// the mixed plan runs j whole rounds of them on the first rows (or columns) of C, data-parallel,
// then the remaining rows (or columns) as a call of their own (split-K, hybrid or
// data-parallel, as planned for that shape).  Same box, three runs each, us, plan for the whole
// matrix -> mixed: 4096 x 11008 x 4096 1802 -> 1730, 11008 x 4096 x 4096 1716 -> 1653, 8192 x 11008
// x 4096 3410 -> 3130, 3072 x 11008 x 4096 1204 -> 1178, 4096 x 14336 x 4096 2205 -> 2030, 2048 x
// 11008 x 4096 888 -> 823, 8192 x 11008 x 1024 895 -> 824, 4352 x 4352 x 1024 225 -> 191, x 4096
// 694 -> 682, 6000 x 6000 x 2048 675 -> 670, 4864 x 4096 x 4096 712 both; two of the thirteen that
// the model takes lose, 4096 x 11008 x 1024 414 -> 431 and 7168 x 4096 x 2048 530 -> 562, whose
// whole-matrix plan runs 6% under its model.  Chosen when the model puts it 1% ahead; the split
// runs along rows or columns, with j from 1 to the whole rounds available.  Only the first level
// splits: the rest is planned without the mixed plan.
// The second launch's fixed cost in the model: its prologue, the first launch's last C stores
// that nothing overlaps, and the gap between the launches (16 us fitted the f32 instruction's
// kernels; 10 us is that at the present rates, and no constant parts the two from the eleven).
constexpr double kMixFixedUs = 10.0;

struct MixPlan {
  int axis = -1;  // 0: rows [0, split) first; 1: columns [0, split) first
  int split = 0;
};

bool mix_plan(int batch, int m, int n, int k, MixPlan& out) {
  if (batch != 1 || k <= 0 || k % kBK != 0) return false;
  const long long cu = bch::device_cu_count();
  const int mt = (m + 255) / 256, nt = (n + 255) / 256;
  const long long rounds = (long long)mt * nt / cu;
  if (rounds < 1) return false;
  const double nk = k / kBK;
  double best = 0.99 * tile_path_cost_us(m, n, k);
  bool found = false;
  for (int axis = 0; axis < 2; ++axis) {
    const int along = axis == 0 ? mt : nt, across = axis == 0 ? nt : mt;
    for (long long j = rounds; j >= 1; --j) {
      const long long c = j * cu / across;  // whole tile rows (columns) that fit j rounds
      if (c < 1 || c >= along) continue;
      const int split = (int)(256 * c);
      const double first = (double)((c * across + cu - 1) / cu) * nk * kTileKtUs;
      const double rest = axis == 0 ? tile_path_cost_us(m - split, n, k) : tile_path_cost_us(m, n - split, k);
      const double cost = first + rest + kMixFixedUs;
      if (cost < best) {
        best = cost;
        found = true;
        out.axis = axis;
        out.split = split;
      }
    }
  }
  return found;
}

// C[tile j's rows and columns] = act(sum over s < S of P[s][j] (+ bias)) for the r split
// tiles j (logical tiles tile0 + j, in the kernel's grouped order); V: four columns per
// thread (N % 4 == 0, ldc % 4 == 0, C and bias 16-byte aligned)
template <bool V, int BM, int BN>
__global__ __launch_bounds__(256) void sgemm_tail_reduce(int M, int N, int tiles_m, int tiles_n, int tile0, int r,
                                                         int S, const float* __restrict__ P, float* __restrict__ C,
                                                         int ldc, const float* __restrict__ bias, int act) {
  constexpr int TS = BM * BN;
  constexpr int w = V ? 4 : 1;
  const long long total = (long long)r * TS / w;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    const long long e = i * w;
    const int j = (int)(e / TS), l = (int)(e - (long long)j * TS);
    const int lr = l / BN, lc = l - lr * BN;
    const int L = tile0 + j, group_size = 8 * tiles_n, g = L / group_size, first_m = g * 8;
    const int gm = min(tiles_m - first_m, 8), within = L - g * group_size;
    const int row = (first_m + within % gm) * BM + lr, col = (within / gm) * BN + lc;
    if (row >= M || col >= N) continue;
    const float* src = P + (long long)j * TS + l;
    if constexpr (V) {
      float4 acc = *reinterpret_cast<const float4*>(src);
      for (int s = 1; s < S; ++s) {
        const float4 x = *reinterpret_cast<const float4*>(src + (long long)s * r * TS);
        acc.x += x.x;
        acc.y += x.y;
        acc.z += x.z;
        acc.w += x.w;
      }
      if (bias) {
        acc.x += bias[col];
        acc.y += bias[col + 1];
        acc.z += bias[col + 2];
        acc.w += bias[col + 3];
      }
      acc = make_float4(bch::activate(acc.x, act), bch::activate(acc.y, act), bch::activate(acc.z, act),
                        bch::activate(acc.w, act));
      *reinterpret_cast<float4*>(C + (long long)row * ldc + col) = acc;
    } else {
      float acc = src[0];
      for (int s = 1; s < S; ++s) acc += src[(long long)s * r * TS];
      if (bias) acc += bias[col];
      C[(long long)row * ldc + col] = bch::activate(acc, act);
    }
  }
}

template <int BM, int BN>
hipError_t launch_tail_reduce(hipStream_t s, int m, int n, const HybPlan& h, const float* P, float* C, int ldc,
                              const float* bias, int act) {
  const int tm = (m + BM - 1) / BM, tn = (n + BN - 1) / BN;
  const bool v = n % 4 == 0 && ldc % 4 == 0 && aligned16(C) && (bias == nullptr || aligned16(bias));
  const long long work = (long long)h.r * BM * BN / (v ? 4 : 1);
  const int blocks = (int)std::min<long long>((work + 255) / 256, 4096);
  if (v)
    hipLaunchKernelGGL((sgemm_tail_reduce<true, BM, BN>), dim3(blocks), dim3(256), 0, s, m, n, tm, tn, h.ndp, h.r,
                       h.S, P, C, ldc, bias, act);
  else
    hipLaunchKernelGGL((sgemm_tail_reduce<false, BM, BN>), dim3(blocks), dim3(256), 0, s, m, n, tm, tn, h.ndp, h.r,
                       h.S, P, C, ldc, bias, act);
  return hipGetLastError();
}

// mode 0: unguarded; mode 1: guarded, 16-byte aligned rows
template <bool TB, bool EPI>
hipError_t launch_hyb(int mode, const HybPlan& h, hipStream_t s, int m, int n, int k, const float* A, int lda,
                      const float* B, int ldb, float* C, int ldc, const float* bias, int act, float* P) {
#define BCH_HYB(BM_, BN_)                                                                                         \
  (mode == 0 ? launch_hyb_tiles<BM_, BN_, kBK, false, TB, EPI, false>(s, m, n, k, A, lda, B, ldb, C, ldc,  \
                                                                            bias, act, h.ndp, h.r, h.S, h.kt, P) \
             : launch_hyb_tiles<BM_, BN_, kBK, true, TB, EPI, true>(s, m, n, k, A, lda, B, ldb, C, ldc, bias, \
                                                                         act, h.ndp, h.r, h.S, h.kt, P))
  hipError_t e = h.t == Tile::k256x256   ? BCH_HYB(256, 256)
                 : h.t == Tile::k256x128 ? BCH_HYB(256, 128)
                                         : BCH_HYB(128, 128);
#undef BCH_HYB
  if (e != hipSuccess) return e;
  return h.t == Tile::k256x256   ? launch_tail_reduce<256, 256>(s, m, n, h, P, C, ldc, bias, act)
         : h.t == Tile::k256x128 ? launch_tail_reduce<256, 128>(s, m, n, h, P, C, ldc, bias, act)
                                 : launch_tail_reduce<128, 128>(s, m, n, h, P, C, ldc, bias, act);
}

// ---- small outputs: 32 x 32 tiles, k over the eight wavefronts of a workgroup ----
// A product of few tiles and short k is latency: launch, one trip to memory, the sums, the store.
// A wavefront takes every eighth 32-k unit of its workgroup's tile, loads the operands straight
// into the MFMA's layout (no LDS, no barrier until the end) with the next unit in flight, and
// the eight blocks are added in wavefront order through LDS: no partials in memory, no reduce
// launch.  Each operand value is read and split once per 32 rows or columns, so larger outputs are
// better off on the split plan's tiles (small_k_plan).
template <bool TB, bool ALIGNED>
__global__ __launch_bounds__(512, 4) void sgemm_small_kernel(int M, int N, int K, const float* __restrict__ A, int lda,
                                                             long long sA, const float* __restrict__ B, int ldb,
                                                             long long sB, float* __restrict__ C, int ldc,
                                                             long long sC, int tiles_m,
                                                             const float* __restrict__ bias, int act) {
  constexpr int W = 8;
  __shared__ float part[W][1024];
  // an XCD's workgroups run neighbouring tiles, a column panel of B at a time
  int lt = blockIdx.x;
  const int nt = gridDim.x;
  if ((nt & 7) == 0) lt = (lt & 7) * (nt >> 3) + (lt >> 3);
  const int m0 = lt % tiles_m * 32, n0 = lt / tiles_m * 32;
  A += blockIdx.y * sA;
  B += blockIdx.y * sB;
  C += blockIdx.y * sC;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, lh = lane >> 5;
  const int row = min(m0 + li, M - 1), col = min(n0 + li, N - 1);
  const float* const pa = A + (long long)row * lda;
  const float* const pb = TB ? B + (long long)col * ldb : B + col;
  const unsigned vb = 4u * (8u * lh * (unsigned)ldb + col);  // [k][n]: this lane's byte offset from a scalar row

  // unit u: k 32 u .. + 31, as two octets of this lane's row and column, 32 u + 16 s + 8 lh ..
  auto load = [&](int u, float (&a)[2][8], float (&b)[2][8]) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      load8<ALIGNED>(pa + 32 * u + 16 * s + 8 * lh, a[s]);
      if constexpr (TB) {
        load8<ALIGNED>(pb + 32 * u + 16 * s + 8 * lh, b[s]);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          b[s][e] = *reinterpret_cast<const float*>(
              reinterpret_cast<const char*>(B + (long long)(32 * u + 16 * s + e) * ldb) + vb);
      }
    }
  };
  auto load_rest = [&](int u, float (&a)[2][8], float (&b)[2][8]) {  // the k remainder: zeros from K on
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int k = 32 * u + 16 * s + 8 * lh + e, kc = min(k, K - 1);
        const float x = pa[kc], y = TB ? pb[kc] : pb[(long long)kc * ldb];
        a[s][e] = k < K ? x : 0.0f;
        b[s][e] = k < K ? y : 0.0f;
      }
  };
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  auto multiply = [&](const float (&a)[2][8], const float (&b)[2][8]) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      u32x4 fa[3], fb[3];
      split8(a[s], fa);
      split8(b[s], fb);
#pragma unroll
      for (int q = 0; q < 6; ++q) acc = bf16_mm(fa[bch::kPartA[q]], fb[bch::kPartB[q]], acc);
    }
  };
  // wavefront w: units w, w + W, ..., its share of the remainder first
  const int nf = K / 32, nu = (K + 31) / 32;
  float a0[2][8], b0[2][8], a1[2][8], b1[2][8];
  int u = wave;
  bool more = true;
  if (nf < nu && wave == nf % W) {
    load_rest(nf, a0, b0);
  } else if (u < nf) {
    load(u, a0, b0);
    u += W;
  } else {
    more = false;
  }
  while (more) {
    if ((more = u < nf)) load(u, a1, b1);
    multiply(a0, b0);
    if (!more) break;
    u += W;
    if ((more = u < nf)) load(u, a0, b0);
    multiply(a1, b1);
    u += W;
  }

  // ---- scaled back; values that are not finite again in f32, this wavefront's units ----
  acc *= bch::kSplitUnscale;
  unsigned want;
  if (non_finite<1, 1>(&acc, &want)) {
    const float* const qb[1] = {pb};
    f32x16 sum[1];
    redo_f32<1, TB>(want, 2 * ((nf - wave + W - 1) / W), [&](int c) { return 32 * (wave + W * (c >> 1)) + 16 * (c & 1); },
                    wave == nf % W ? 32 * nf : K, K, lh, pa, qb, ldb, sum);
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = want >> r & 1u ? sum[0][r] : acc[r];
  }

  // ---- the eight blocks added in wavefront order, two values a thread ----
#pragma unroll
  for (int r = 0; r < 16; ++r) part[wave][64 * r + lane] = acc[r];
  __syncthreads();
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int i = tid + 512 * h, r = i >> 6;
    float v = part[0][i];
#pragma unroll
    for (int w = 1; w < W; ++w) v += part[w][i];
    const int om = m0 + 8 * (r >> 2) + 4 * lh + (r & 3), on = n0 + li;
    if (om < M && on < N) C[(long long)om * ldc + on] = bch::activate(v + (bias ? bias[on] : 0.0f), act);
  }
}

// Modelled us: a workgroup's pass of 256 k takes 1.35 us of its CU, alone on it or not, next to
// 3.2 us of launch, first loads and store, against the split plan's model, which is 2 to 5 us low at
// these sizes.  Measured, one box, us, before -> here: 65^3 7.5 -> 4.5, 300^3 11.8 -> 5.0, 171 x 455 x 1472
// 15.0 -> 11.4, 100 x 4000 x 500 15.5 -> 9.6, 1001 x 999 x 333 17.9 -> 13.1, 256 x 1024 x 1024 (split) 15.8 -> 8.5,
// 512 x 512 x 1024 15.8 -> 9.0; left to the split plan: 700 x 1200 x 1500 26.6 (38.2 here), 256 x 2048 x
// 2048 22.9 (24.6).  From k 2048 on the split plan's shorter sums are the more exact (128 x 128 x 2048
// 1.9e-7 against 2.5e-7) and the times within 15%.  Below 64 k the tiles stay, which multiply in
// f32 below one pass of theirs (a lone product rounds once there, and is up to 2.0 2^-24 off as part
// products); 100 x 4000 x 48 takes 7.6 us on them.
bool small_k_plan(int batch, int m, int n, int k) {
  if (batch < 1 || batch > 65535 || k < 64 || k >= 2048) return false;
  const SplitPlan p = split_plan(batch, m, n, k);
  if (p.us == 0.0) return false;  // whole rounds of the other tiles
  const long long cu = bch::device_cu_count();
  const long long wgs = (long long)batch * ((m + 31) / 32) * ((n + 31) / 32);
  return 3.2 + 1.35 * (double)((wgs + cu - 1) / cu) * ((k + 255) / 256) < p.us + 2.0;
}

// the kernel's byte offsets of 8 rows of a [k][n] B and a column stay below 2^32
bool small_k_ok(int batch, int m, int n, int k, int ldb) {
  return ldb < (1 << 26) && small_k_plan(batch, m, n, k);
}

hipError_t launch_small_k(hipStream_t s, bool transb, int batch, int m, int n, int k, const float* A, int lda,
                          long long sA, const float* B, int ldb, long long sB, const float* bias, int act, float* C,
                          int ldc, long long sC) {
  const int tm = (m + 31) / 32, tn = (n + 31) / 32;
  const bool a16 = aligned16(A) && lda % 4 == 0 && (batch == 1 || sA % 4 == 0);
  const bool b16 = aligned16(B) && ldb % 4 == 0 && (batch == 1 || sB % 4 == 0);
#define BCH_SMALL_K(TB_, AL_)                                                                                    \
  hipLaunchKernelGGL((sgemm_small_kernel<TB_, AL_>), dim3(tm * tn, batch), dim3(512), 0, s, m, n, k, A, lda, sA, \
                     B, ldb, sB, C, ldc, sC, tm, bias, act)
  if (transb) {
    if (a16 && b16) BCH_SMALL_K(true, true); else BCH_SMALL_K(true, false);
  } else {
    if (a16) BCH_SMALL_K(false, true); else BCH_SMALL_K(false, false);
  }
#undef BCH_SMALL_K
  return hipGetLastError();
}

// ---- few rows: 32 or 64 x 128 tiles, k split over the chip (the rows kernel) ----
// Up to 64 rows against [n][k] weights, or [k][n] weights that the skinny kernels do not take: the
// job is streaming B once.  A workgroup owns 128 columns and one k-slice; its 512 threads load an
// octet of B each per 32-k pass, two passes in flight (64 KB a CU with two workgroups), and
// put the three parts into LDS as the large tiles do; four wavefronts side by side take 32 columns
// each, a second set of four the other 16 k of the pass, so each wavefront runs 6 MFMAs per 32
// rows and pass.  The slices' partials meet in sgemm_splitk_reduce.  At 32 rows the matrix work is
// 7 us of the 29 us that 4096 x 11008 weights take to stream (18 us as v_mfma_f32_32x32x2_f32).
// Measured (one box, us, MLP of [n][k] weights with bias and GELU, before -> now): 48 rows 4096 ->
// 11008 -> 4096 175 -> 117, 32 rows 4095 -> 11007 -> 4095 1364 -> 116, 2 rows 640 -> 8001 -> 640
// 738 -> 50.  It streams at 4.1 TB/s: conversion, LDS traffic and MFMAs of a pass each take 400 to
// 600 cycles and overlap only between the two workgroups.
template <int TM>
struct RowsCfg {
  static constexpr int BN = 128, KS = 32, NO = KS / 8, NT = 512;
  static constexpr int ASTR = 32 * TM * 16 + 32, BSTR = BN * 16 + 32;  // bytes of one octet of one part
  static constexpr int ABYTES = 3 * NO * ASTR, BUF = ABYTES + 3 * NO * BSTR;
};

template <int TM, bool TB>
__global__ __launch_bounds__(512, 4) void sgemm_rows_kernel(int M, int N, int K, const float* __restrict__ A, int lda,
                                                            const float* __restrict__ B, int ldb, float* __restrict__ C,
                                                            int ldc, long long sC, const float* __restrict__ bias,
                                                            int act, int kc) {
  using G = RowsCfg<TM>;
  constexpr int KS = G::KS, NO = G::NO;
  __shared__ __attribute__((aligned(16))) char lds[2 * G::BUF];
  const int n0 = blockIdx.x * G::BN, z = blockIdx.y;
  A += (long long)z * kc;
  B += TB ? (long long)z * kc : (long long)z * kc * ldb;
  C += z * sC;
  K = min(kc, K - z * kc);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, lh = lane >> 5;
  const int kg = wave >> 2, wn = (wave & 3) * 32;
  const bool a_wave = wave < 2 * TM;  // these load A's octets too

  const float* pa = A + (long long)min(tid / NO, M - 1) * lda + 8 * (tid % NO);
  const int brow = TB ? tid / NO : tid % G::BN, boct = TB ? tid % NO : wave >> 1;
  const int bcol = min(n0 + brow, N - 1);
  const float* pb = TB ? B + (long long)bcol * ldb + 8 * boct : B + (long long)(8 * boct) * ldb;
  float ra[2][8], rb[2][8];
  auto load = [&](int set, int k0) {
    if (a_wave) load8<false>(pa + k0, ra[set]);
    if constexpr (TB) {
      load8<false>(pb + k0, rb[set]);
    } else {
      const float* s = pb + (long long)k0 * ldb;
#pragma unroll
      for (int e = 0; e < 8; ++e) rb[set][e] = s[(long long)e * ldb + (unsigned)bcol];
    }
  };
  auto load_rest = [&](int k0) {  // zeros from K on
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int ka = k0 + 8 * (tid % NO) + e, kb = k0 + 8 * boct + e;
      const int da = min(ka, K - 1) - 8 * (tid % NO), db = min(kb, K - 1) - 8 * boct;
      const float x = a_wave ? pa[da] : 0.0f, y = TB ? pb[db] : pb[(long long)db * ldb + bcol];
      ra[0][e] = ka < K ? x : 0.0f;
      rb[0][e] = kb < K ? y : 0.0f;
    }
  };
  auto store = [&](int buf, int set) {
    char* s = lds + buf * G::BUF;
    u32x4 q[3];
    if (a_wave) {
      split8(ra[set], q);
#pragma unroll
      for (int p3 = 0; p3 < 3; ++p3)
        *reinterpret_cast<u32x4*>(s + (p3 * NO + tid % NO) * G::ASTR + (tid / NO) * 16) = q[p3];
    }
    split8(rb[set], q);
#pragma unroll
    for (int p3 = 0; p3 < 3; ++p3)
      *reinterpret_cast<u32x4*>(s + G::ABYTES + (p3 * NO + boct) * G::BSTR + brow * 16) = q[p3];
  };
  f32x16 acc[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
  auto multiply = [&](int buf) {
    const char* s = lds + buf * G::BUF;
    u32x4 fa[TM][3], fb[3];
#pragma unroll
    for (int p3 = 0; p3 < 3; ++p3) {
      const int oct = p3 * NO + 2 * kg + lh;
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[i][p3] = *reinterpret_cast<const u32x4*>(s + oct * G::ASTR + (32 * i + li) * 16);
      fb[p3] = *reinterpret_cast<const u32x4*>(s + G::ABYTES + oct * G::BSTR + (wn + li) * 16);
    }
#pragma unroll
    for (int q = 0; q < 6; ++q)
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[i] = bf16_mm(fa[i][bch::kPartA[q]], fb[bch::kPartB[q]], acc[i]);
  };

  // pass t: parts of pass t + 1 to the other buffer, loads of pass t + 3, products of pass t
  const int nk = (K + KS - 1) / KS, rest = K % KS != 0 ? 1 : 0;  // a remainder runs first
  auto k_of = [&](int t) { return (min(t, nk - 1) - rest) * KS; };
  if (rest)
    load_rest((nk - 1) * KS);
  else
    load(0, 0);
  store(0, 0);
  if (nk > 1) {
    load(1, k_of(1));
    load(0, k_of(2));
  }
  __syncthreads();
  int t = 0;
  for (; t + 2 < nk; t += 2) {
    store(1, 1);
    load(1, k_of(t + 3));
    multiply(0);
    __syncthreads();
    store(0, 0);
    load(0, k_of(t + 4));
    multiply(1);
    __syncthreads();
  }
  if (t + 1 < nk) {
    store(1, 1);
    multiply(0);
    __syncthreads();
    multiply(1);
  } else {
    multiply(0);
  }

  // ---- the two halves of k added up ----
  const int col = n0 + wn + li;
  __syncthreads();  // the last pass's reads are done
  f32x16* const part = reinterpret_cast<f32x16*>(lds) + (wave & 3) * (64 * TM) + lane;
  if (kg != 0) {
#pragma unroll
    for (int i = 0; i < TM; ++i) part[64 * i] = acc[i];
  }
  __syncthreads();
  if (kg != 0) return;
#pragma unroll
  for (int i = 0; i < TM; ++i) acc[i] = (acc[i] + part[64 * i]) * bch::kSplitUnscale;
  unsigned want[TM];
  const bool redo = non_finite<TM, 1>(acc, want);
  const float bj = bias && col < N ? bias[col] : 0.0f;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = 32 * i + 8 * (r >> 2) + 4 * lh + (r & 3);
      if (row < M && col < N) C[(long long)row * ldc + col] = bch::activate(acc[i][r] + bj, act);
    }
  if (!redo) return;
#pragma unroll 1
  for (int i = 0; i < TM; ++i) {  // as for the large tiles: again in f32, after the stores
    const unsigned w = i == 0 ? want[0] : want[TM - 1];
    if (!__any(w != 0)) continue;
    const float* const qb[1] = {TB ? B + (long long)min(col, N - 1) * ldb : B + min(col, N - 1)};
    f32x16 sum[1];
    redo_f32<1, TB>(w, K / 16, [](int c) { return 16 * c; }, K / 16 * 16, K, lh,
                       A + (long long)min(32 * i + li, M - 1) * lda, qb, ldb, sum);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = 32 * i + 8 * (r >> 2) + 4 * lh + (r & 3);
      if ((w >> r & 1u) && row < M && col < N) C[(long long)row * ldc + col] = bch::activate(sum[0][r] + bj, act);
    }
  }
}

// Two workgroups per CU resident at once, slices of 4 passes or more; the partials stay under the
// small scratch, so bch_sgemm_noalloc and bch_sgemm plan alike.
struct RowsPlan {
  int S = 1, kc = 0;
};
RowsPlan rows_plan(int m, int n, int k) {
  RowsPlan p;
  const int tiles = (n + 127) / 128, nk = (k + 31) / 32;
  long long s = 2LL * bch::device_cu_count() / tiles;
  s = std::min<long long>({s, nk / 4, (long long)(kSplitWsSmall / (sizeof(float) * (size_t)m * n))});
  if (s < 1) s = 1;
  p.kc = (int)((nk + s - 1) / s) * 32;
  p.S = (k + p.kc - 1) / p.kc;
  return p;
}
// Up to 64 rows where no skinny kernel takes the call (its K, N or alignment: against the tile
// path's slices MLP of 20 rows 2890 -> 5248 53 -> 46 us), and 33 to 64 rows against [n][k]
// weights too large for the tile path's slices to stay in step (in us, two passes of the 32-row
// kernels or tile slices -> here: 48 x 11008 x 4096 78 -> 55, 64 x 4096 x 11008 75 -> 59, 48 x
// 4096 x 1024 17.7 -> 16.9; 48 x 5120 x 2048 23.0 -> 24.2, so from 2^24 weights on).  Two passes of
// the 32-row kernels lose to both below that too (48 x 11008 x 1024 31.7, tile path 27.0, here 24.4;
// 40 x 32768 x 256 185, 15.7, 20.0; 64 x 8192 x 1024 30.4, 16.4, 22.9).
bool rows_applies(bool transb, int batch, int m, int n, int k, const float* A, int lda, const float* B, int ldb) {
  if (batch != 1 || m > 64 || n < 1 || k < 1) return false;
  if (transb)
    return m > 32 ? (long long)n * k >= (1LL << 24) || k % 4 != 0
                  : !bch::sgemm_skinny_nt_applies(m, n, k, A, lda, B, ldb);
  return !bch::sgemm_skinny_applies(m, n, k, A, lda, B, ldb) && (m <= 32 || n % 4 != 0);
}
size_t rows_bytes(int m, int n, int k) {
  const RowsPlan p = rows_plan(m, n, k);
  return p.S > 1 ? (size_t)p.S * m * n * sizeof(float) : 0;
}

hipError_t launch_rows(hipStream_t s, bool transb, int m, int n, int k, const float* A, int lda, const float* B,
                       int ldb, float* C, int ldc, const float* bias, int act, void* ws) {
  const RowsPlan p = rows_plan(m, n, k);
  const bool split = p.S > 1;
  float* out = split ? static_cast<float*>(ws) : C;
  const dim3 grid((n + 127) / 128, p.S);
#define BCH_ROWS(TM_, TB_)                                                                                       \
  hipLaunchKernelGGL((sgemm_rows_kernel<TM_, TB_>), grid, dim3(512), 0, s, m, n, k, A, lda, B, ldb, out,          \
                     split ? n : ldc, split ? (long long)m * n : 0LL, split ? nullptr : bias, split ? 0 : act, p.kc)
  if (m <= 32) {
    if (transb) BCH_ROWS(1, true); else BCH_ROWS(1, false);
  } else {
    if (transb) BCH_ROWS(2, true); else BCH_ROWS(2, false);
  }
#undef BCH_ROWS
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !split) return e;
  return launch_splitk_reduce(s, m, n, p.S, 1, static_cast<const float*>(ws), C, ldc, 0, bias, act);
}

}  // namespace

namespace bch {

static const char* tile_path_name(int m, int n, int k, bool allow_mix);

const char* sgemm_kernel_name(int m, int n, int k) {
  if (sgemm_skinny_applies(m, n, k, nullptr, k, nullptr, n)) return sgemm_skinny_kernel_name(m);
  if (rows_applies(false, 1, m, n, k, nullptr, k, nullptr, n)) {
    static const char* const names[2][2] = {{"sgemm_rows_kernel<1>", "sgemm_rows_kernel<1>+sgemm_splitk_reduce"},
                                            {"sgemm_rows_kernel<2>", "sgemm_rows_kernel<2>+sgemm_splitk_reduce"}};
    return names[m > 32][rows_plan(m, n, k).S > 1];
  }
  return tile_path_name(m, n, k, true);
}

// The tile path's kernels for lda = k, ldb = n and 16-byte aligned operands.
static const char* tile_path_name(int m, int n, int k, bool allow_mix) {
  MixPlan mp;
  if (allow_mix && mix_plan(1, m, n, k, mp)) {
    const int m1 = mp.axis == 0 ? mp.split : m, n1 = mp.axis == 1 ? mp.split : n;
    const bool fast = m1 % 256 == 0 && n1 % 256 == 0 && n % 4 == 0;
    thread_local std::string name;
    name = std::string(fast ? "sgemm_mfma_kernel<256,256,32,false>" : "sgemm_mfma_kernel<256,256,32,true,v4>") +
           (mp.axis == 0 ? " rows then " : " columns then ") +
           (mp.axis == 0 ? tile_path_name(m - m1, n, k, false) : tile_path_name(m, n - n1, k, false));
    return name.c_str();
  }
  if (small_tile_plan(1, m, n, k)) return "sgemm_mfma_kernel<64,64,64,false>";
  if (small_k_ok(1, m, n, k, n)) return "sgemm_small_kernel";
  const SplitPlan sp = split_plan(1, m, n, k);
  const Tile t = sp.S > 1 ? sp.t : pick_tile(1, m, n);
  // with lda = k and ldb = n, and 16-byte aligned operands
  const bool check = !(m % tile_m(t) == 0 && n % tile_n(t) == 0 && k % kBK == 0 && k % 4 == 0 && n % 4 == 0);
  const bool v4 = k >= 4 && k % 4 == 0 && n % 4 == 0;
  if (sp.S > 1) {
    const bool fast = !check;
    static const char* const split_names[3][3] = {
        {"sgemm_mfma_kernel<256,256,32,false>+sgemm_splitk_reduce", "sgemm_mfma_kernel<256,256,32,true,v4>+sgemm_splitk_reduce",
         "sgemm_mfma_kernel<256,256,32,true>+sgemm_splitk_reduce"},
        {"sgemm_mfma_kernel<256,128,32,false>+sgemm_splitk_reduce", "sgemm_mfma_kernel<256,128,32,true,v4>+sgemm_splitk_reduce",
         "sgemm_mfma_kernel<256,128,32,true>+sgemm_splitk_reduce"},
        {"sgemm_mfma_kernel<128,128,32,false>+sgemm_splitk_reduce", "sgemm_mfma_kernel<128,128,32,true,v4>+sgemm_splitk_reduce",
         "sgemm_mfma_kernel<128,128,32,true>+sgemm_splitk_reduce"}};
    return split_names[static_cast<int>(t)][fast ? 0 : v4 ? 1 : 2];
  }
  HybPlan h;
  if (hyb_plan(1, m, n, k, h)) {
    const bool fast = m % tile_m(h.t) == 0 && n % tile_n(h.t) == 0 && n % 4 == 0;
    static const char* const hyb_names[3][2] = {
        {"sgemm_mfma_kernel<256,256,32,false,hyb>+sgemm_tail_reduce", "sgemm_mfma_kernel<256,256,32,true,v4,hyb>+sgemm_tail_reduce"},
        {"sgemm_mfma_kernel<256,128,32,false,hyb>+sgemm_tail_reduce", "sgemm_mfma_kernel<256,128,32,true,v4,hyb>+sgemm_tail_reduce"},
        {"sgemm_mfma_kernel<128,128,32,false,hyb>+sgemm_tail_reduce", "sgemm_mfma_kernel<128,128,32,true,v4,hyb>+sgemm_tail_reduce"}};
    if (fast || v4) return hyb_names[static_cast<int>(h.t)][fast ? 0 : 1];
  }
  return tile_name(t, !check ? 0 : v4 ? 1 : 2);
}

// The tile path's scratch: split-K partials, or the hybrid plan's.
static size_t tile_workspace_bytes(int batch, int m, int n, int k, bool allow_mix = true) {
  MixPlan mp;
  if (allow_mix && mix_plan(batch, m, n, k, mp))  // the whole tiles need none; the rest is a call of its own
    return mp.axis == 0 ? tile_workspace_bytes(1, m - mp.split, n, k, false)
                        : tile_workspace_bytes(1, m, n - mp.split, k, false);
  const int sl = split_slices(batch, m, n, k);
  if (sl > 1) return (size_t)sl * batch * m * n * sizeof(float);
  HybPlan h;
  return hyb_plan(batch, m, n, k, h) ? hyb_bytes(h) : 0;
}

size_t sgemm_workspace_bytes(int batch, int m, int n, int k) {
  if (batch == 1 && sgemm_skinny_applies(m, n, k, nullptr, k, nullptr, n))
    return sgemm_skinny_workspace_bytes(m, n, k);
  return tile_workspace_bytes(batch, m, n, k);
}

size_t sgemm_ex_workspace_bytes(bool transb, int batch, int m, int n, int k, const float* A, int lda, long long sA,
                                const float* B, int ldb, long long sB) {
  if (rows_applies(transb, batch, m, n, k, A, lda, B, ldb)) return rows_bytes(m, n, k);
  if (batch == 1 && !transb && sgemm_skinny_applies(m, n, k, nullptr, k, nullptr, n))
    return sgemm_skinny_workspace_bytes(m, n, k);
  if (batch == 1 && sgemm_skinny_nt_applies(m, n, k, nullptr, lda, nullptr, ldb))
    return sgemm_skinny_nt_workspace_bytes(m, n, k);
  if (small_tile_ok(batch, m, n, k, A, lda, sA, B, ldb, sB) || small_k_ok(batch, m, n, k, ldb)) return 0;
  return tile_workspace_bytes(batch, m, n, k);
}

hipError_t launch_sgemm(hipStream_t s, int batch, int m, int n, int k, const float* A, int lda, long long sA,
                        const float* B, int ldb, long long sB, float* C, int ldc, long long sC, void* ws,
                        size_t ws_bytes) {
  return launch_sgemm_ex(s, false, batch, m, n, k, A, lda, sA, B, ldb, sB, nullptr, 0, C, ldc, sC, ws, ws_bytes);
}

}  // namespace bch

namespace {

// The tile path of launch_sgemm_ex: split-K, the mixed plan (allow_mix), the hybrid plan or the
// data-parallel tiling.
hipError_t launch_tile_path(hipStream_t s, bool transb, int batch, int m, int n, int k, const float* A, int lda,
                            long long sA, const float* B, int ldb, long long sB, const float* bias, int act,
                            float* C, int ldc, long long sC, void* ws, size_t ws_bytes, bool allow_mix);

}  // namespace

namespace bch {

hipError_t launch_sgemm_ex(hipStream_t s, bool transb, int batch, int m, int n, int k, const float* A, int lda,
                           long long sA, const float* B, int ldb, long long sB, const float* bias, int act,
                           float* C, int ldc, long long sC, void* ws, size_t ws_bytes) {
  if (batch <= 0 || m <= 0 || n <= 0) return hipSuccess;
  // m <= 32: the skinny kernels always (their partials sized by the caller); 32 < m <= 64:
  // the 64-row skinny kernel when its partials fit the scratch at hand, else the tiles
  if (!transb && batch == 1 && sgemm_skinny_applies(m, n, k, A, lda, B, ldb) &&
      (m <= 32 || (ws != nullptr && ws_bytes >= sgemm_skinny_workspace_bytes(m, n, k))))
    return launch_sgemm_skinny(s, m, n, k, A, lda, B, ldb, C, ldc, ws, ws_bytes, bias, act);
  if (transb && batch == 1 && sgemm_skinny_nt_applies(m, n, k, A, lda, B, ldb))
    return launch_sgemm_skinny_nt(s, m, n, k, A, lda, B, ldb, C, ldc, ws, ws_bytes, bias, act);
  if (rows_applies(transb, batch, m, n, k, A, lda, B, ldb) && ws_bytes >= rows_bytes(m, n, k))
    return launch_rows(s, transb, m, n, k, A, lda, B, ldb, C, ldc, bias, act, ws);
  return launch_tile_path(s, transb, batch, m, n, k, A, lda, sA, B, ldb, sB, bias, act, C, ldc, sC, ws, ws_bytes,
                          true);
}

}  // namespace bch

namespace {

hipError_t launch_tile_path(hipStream_t s, bool transb, int batch, int m, int n, int k, const float* A, int lda,
                            long long sA, const float* B, int ldb, long long sB, const float* bias, int act,
                            float* C, int ldc, long long sC, void* ws, size_t ws_bytes, bool allow_mix) {
  if (small_tile_ok(batch, m, n, k, A, lda, sA, B, ldb, sB)) {
    const bool epi = bias != nullptr || act != 0;
#define BCH_SMALL(TB_, EPI_)                                                                                       \
  launch_tiles<64, 64, kSmallBK, false, TB_, EPI_>(s, batch, m, n, k, A, lda, sA, B, ldb, sB, C, ldc, sC, bias, act)
    return transb ? (epi ? BCH_SMALL(true, true) : BCH_SMALL(true, false))
                  : (epi ? BCH_SMALL(false, true) : BCH_SMALL(false, false));
#undef BCH_SMALL
  }
  if (small_k_ok(batch, m, n, k, ldb))
    return launch_small_k(s, transb, batch, m, n, k, A, lda, sA, B, ldb, sB, bias, act, C, ldc, sC);
  SplitPlan sp = split_plan(batch, m, n, k);
  const size_t pbytes = (size_t)batch * m * n * sizeof(float);  // one slice's partials, every batch
  if (sp.S > 1 && (ws == nullptr || ws_bytes < (size_t)sp.S * pbytes))
    sp = split_plan(batch, m, n, k, ws == nullptr ? 0 : ws_bytes);  // fewer slices within the scratch at hand
  const Tile t = sp.S > 1 ? sp.t : pick_tile(batch, m, n);
  const int sl = sp.S;
  if (sl > 1 && ws != nullptr && ws_bytes >= (size_t)sl * pbytes) {
    // batch b, slice j (grid.z): A + b sA + j kc, B + b sB + j kc rows (columns for [n][k]),
    // into P[b][j] (m x n)
    const int kc = sp.kc;
    float* P = static_cast<float*>(ws);
    const long long per = (long long)m * n;
    ZSplit z;
    z.nz = sl;
    z.kc = kc;
    z.sA = kc;
    z.sB = transb ? (long long)kc : (long long)kc * ldb;
    z.sC = per;
    // the slice offsets (kc a multiple of 32, times ldb) keep the batch strides' alignment
    const int mode = fast_ok(t, m, n, k, A, lda, sA, B, ldb, sB)               ? 0
                     : vec4_ok(n, k, A, lda, sA, B, ldb, sB) ? 1
                                                                           : 2;
    hipError_t e = transb ? launch_tile_any<true, false>(mode, t, s, batch, m, n, k, A, lda, sA, B, ldb, sB, P, n,
                                                         sl * per, nullptr, 0, z)
                          : launch_tile_any<false, false>(mode, t, s, batch, m, n, k, A, lda, sA, B, ldb, sB, P, n,
                                                          sl * per, nullptr, 0, z);
    if (e != hipSuccess) return e;
    return launch_splitk_reduce(s, m, n, sl, batch, P, C, ldc, sC, bias, act);
  }
  const bool epi = bias != nullptr || act != 0;
  MixPlan mp;
  if (allow_mix && mix_plan(batch, m, n, k, mp)) {
    // whole rounds of 256 x 256 tiles on the first rows (columns) of C, then the rest as a call
    // of its own; the offsets are multiples of 256 rows (columns), which keeps the alignment
    const int m1 = mp.axis == 0 ? mp.split : m, n1 = mp.axis == 1 ? mp.split : n;
    const int mode1 = fast_ok(Tile::k256x256, m1, n1, k, A, lda, sA, B, ldb, sB)      ? 0
                      : vec4_ok(n1, k, A, lda, sA, B, ldb, sB) ? 1
                                                                             : 2;
    hipError_t e =
        transb ? (epi ? launch_tile_any<true, true>(mode1, Tile::k256x256, s, 1, m1, n1, k, A, lda, sA, B, ldb, sB, C,
                                                    ldc, sC, bias, act)
                      : launch_tile_any<true, false>(mode1, Tile::k256x256, s, 1, m1, n1, k, A, lda, sA, B, ldb, sB,
                                                     C, ldc, sC, bias, act))
               : (epi ? launch_tile_any<false, true>(mode1, Tile::k256x256, s, 1, m1, n1, k, A, lda, sA, B, ldb, sB,
                                                     C, ldc, sC, bias, act)
                      : launch_tile_any<false, false>(mode1, Tile::k256x256, s, 1, m1, n1, k, A, lda, sA, B, ldb, sB,
                                                      C, ldc, sC, bias, act));
    if (e != hipSuccess) return e;
    if (mp.axis == 0)
      return launch_tile_path(s, transb, 1, m - m1, n, k, A + (long long)m1 * lda, lda, sA, B, ldb, sB, bias, act,
                              C + (long long)m1 * ldc, ldc, sC, ws, ws_bytes, false);
    const float* B2 = transb ? B + (long long)n1 * ldb : B + n1;
    return launch_tile_path(s, transb, 1, m, n - n1, k, A, lda, sA, B2, ldb, sB, bias ? bias + n1 : nullptr, act,
                            C + n1, ldc, sC, ws, ws_bytes, false);
  }
  HybPlan h;
  if (hyb_plan(batch, m, n, k, h) && ws != nullptr && ws_bytes >= hyb_bytes(h)) {
    const int hmode = fast_ok(h.t, m, n, k, A, lda, sA, B, ldb, sB)                ? 0
                      : vec4_ok(n, k, A, lda, sA, B, ldb, sB)          ? 1
                                                                                   : 2;
    if (hmode != 2) {
      float* P = static_cast<float*>(ws);
      if (transb)
        return epi ? launch_hyb<true, true>(hmode, h, s, m, n, k, A, lda, B, ldb, C, ldc, bias, act, P)
                   : launch_hyb<true, false>(hmode, h, s, m, n, k, A, lda, B, ldb, C, ldc, bias, act, P);
      return epi ? launch_hyb<false, true>(hmode, h, s, m, n, k, A, lda, B, ldb, C, ldc, bias, act, P)
                 : launch_hyb<false, false>(hmode, h, s, m, n, k, A, lda, B, ldb, C, ldc, bias, act, P);
    }
  }
  const int mode = fast_ok(t, m, n, k, A, lda, sA, B, ldb, sB) ? 0
                   : vec4_ok(n, k, A, lda, sA, B, ldb, sB) ? 1
                                                                 : 2;
  if (transb)
    return epi ? launch_tile_any<true, true>(mode, t, s, batch, m, n, k, A, lda, sA, B, ldb, sB, C, ldc, sC, bias, act)
               : launch_tile_any<true, false>(mode, t, s, batch, m, n, k, A, lda, sA, B, ldb, sB, C, ldc, sC, bias,
                                              act);
  return epi ? launch_tile_any<false, true>(mode, t, s, batch, m, n, k, A, lda, sA, B, ldb, sB, C, ldc, sC, bias, act)
             : launch_tile_any<false, false>(mode, t, s, batch, m, n, k, A, lda, sA, B, ldb, sB, C, ldc, sC, bias,
                                             act);
}

}  // namespace

// sdpa_fwd.hip -- fused scaled-dot-product attention forward for gfx950.
//
// Replaces the reference's three-pass attention (crates/barracuda/src/ops/
// attention/compute.rs:21-111: K6 shaders/math/attention_matmul_f64.wgsl
// writes the [B,H,Sq,Skv] scores, K7 activation/attention_softmax_f64.wgsl
// normalises them, K9 attention/attention_apply_f64.wgsl multiplies by V),
// its causal variant (ops/causal_attn/compute.rs:24-115 with K8, and the CPU
// ops/causal_attention.rs:52-134) and FlashAttention (ops/flash_attention.rs
// :96-145, K13).  Contract: o[b,h,i,:] = sum_j softmax_j(scale q_i . k_j) v_j,
// j <= i when causal.  The score matrix is never written to memory.
//
// Layout: per tensor a (batch, head, row) stride in elements with the head
// dimension contiguous; [B,H,S,D] row-major is the dense case.  K and V may
// have fewer heads than Q (grouped-query attention, ops/
// grouped_query_attention/compute.rs:27-121): query head h reads key/value
// head h / (H / Hkv).  Strided views also give multi-head attention its
// head split and concat for free (ops/mha/projections.rs:18-58 copy
// [B,S,H*D] <-> [B,H,S,D] through head_split_f64.wgsl / head_concat_f64.wgsl;
// here the kernel reads and writes the [B,S,H,D] projections in place).
//
// Head dimensions: D <= 128 run sdpa_fwd_kernel (below); 128 < D <= 256
// run sdpa_fwd16_kernel (16 queries per wavefront, further down); larger D
// take the chunked three-step path of sdpa_wide.hip.
//
// Design of sdpa_fwd_kernel (both products on the bf16 matrix cores, three exact bf16 parts per
// f32 and six part products accumulated in f32: bch_internal.h, split8):
//   * A workgroup = 8 wavefronts = 256 queries of one (b,h), or 4 = 128 where those would not
//     fill the chip; wavefront w owns queries q0 + 32w .. +31, lane l's query is l % 32.  Key
//     blocks of 32 are split into parts on their way into LDS, once per workgroup,
//     double-buffered, one barrier per block; blocks are loaded two ahead.
//   * What bounds it: per wavefront and block 96 MFMAs of 32 cycles (D = 128) against 256 of 64
//     for v_mfma_f32_32x32x2_f32, next to about 370 VALU operations (softmax, and the parts of
//     P and of its share of K and V); two wavefronts per SIMD overlap the two.  Measured at B 4,
//     H 32, S 2048, D 128, causal, against f32 MFMAs (one box): 1.09 -> 0.71 ms, error against 64
//     bits 4.5e-7 -> 3.7e-7; the matrix cores are busy 57% of the cycles (non-causal 64%), at a
//     clock that has fallen to 1.9 GHz (1.7).
//   * Scores are computed transposed, S^T = K Q^T (32 keys x 32 queries), so
//     each lane holds 16 scores of ITS query: the row max and row sum are
//     in-lane plus one exchange between the two lane halves
//     (v_permlane32_swap).  The q parts stay in registers for the whole kernel (24 registers per
//     32 of D), pre-multiplied by scale*log2(e) so the softmax uses exp2 directly.
//   * The PV product is computed as O^T += V^T P^T, whose B operand is
//     exactly the P values the lane already holds: value r of the S^T block
//     is key 8(r/4) + 4(l/32) + r%4, so 16-k step s contracts keys 16 s + 4 (l/32) + {0..3,
//     8..11}, and V's parts are stored in LDS in that order, [octet][d][8 keys].  P never leaves
//     registers.
//   * Online softmax with a lazily moved reference max: exponentials are
//     taken against a per-query reference m_ref, which only moves (and O and
//     the running sum are only rescaled) when a block's max exceeds it by
//     more than 2^8.  Every term stays <= 256 and the final O / l is exact
//     algebra, so accuracy is unchanged while the rescale of the O accumulator almost never runs.
//   * Causal: key blocks past the workgroup's last query are not loaded;
//     blocks entirely above a wavefront's diagonal are skipped by that
//     wavefront; the diagonal block is masked per element.  Workgroups are
//     issued longest first across all heads (query block major); with
//     B*H % 8 == 0 every query block of a head then lands on one XCD.
//   * Non-causal: workgroups are issued head-major and remapped so that each
//     XCD (dispatch is round-robin over the 8 XCDs) runs a contiguous range
//     of heads, all query blocks of a head together; query heads sharing a
//     key/value head (grouped-query) are adjacent, so they share it in the same L2.
//   * Too few query blocks for the chip: the keys of each are split over workgroups, whose
//     results (unnormalised O, reference max, sum) meet in sdpa_combine (sdpa_decode.hip).
//   * Parts are of 2^16 times the operand (split8); scores are scaled back in the fused
//     multiply-add that subtracts the reference max, O at the end.  Where the scaled numbers may pass
//     f32's range, the wavefront redoes its queries on v_mfma_f32_32x32x2_f32 from global memory:
//     an infinite, NaN or huge V (or a NaN score) leaves a result that is not finite; scores, of
//     which one infinite before its sum ends could pass for a masked one, are bounded by their
//     operands, |q scale log2(e)| and |K| below 2^43, seen while splitting.
#include "bch_internal.h"

#include <math.h>

#include <algorithm>
#include <type_traits>

namespace {

using bch::bf16_mm;
using bch::f32x16;
using bch::split8;
using bch::u32x4;

constexpr int kBKV = 32;  // keys per block
constexpr int kVLD = kBKV + 4;
constexpr float kLog2E = 1.44269504088896340736f;
constexpr float kLazy = 8.0f;  // log2 headroom before the reference max moves
// 128 products of operands below this, scaled by 2^32 (and their leading parts, up to 2^-8 larger),
// stay below 2^127.
constexpr float kScoreBig = 0x1p43f;

// NT threads per workgroup: NT / 64 wavefronts of 32 queries each.
template <int DP, int NT>
struct SdpaCfg {
  static constexpr int BQ = NT / 2;                    // queries per workgroup
  static constexpr int KLD = DP + 4;
  static constexpr int KD4 = DP / 4;                   // float4 per K row
  static constexpr int K_TOT = kBKV * DP / 4;          // float4 of K per tile
  static constexpr int K_F4 = (K_TOT + NT - 1) / NT;    // float4 of K per thread
  static constexpr int V_BLK = kBKV * DP / 16;          // 4x4 V blocks per tile
  static constexpr int V_PER = (V_BLK + NT - 1) / NT;    // 4x4 V blocks per thread
  static constexpr int LDS_FLOATS = 2 * (kBKV * KLD + DP * kVLD);
  static_assert(K_F4 >= 1, "K tile must cover the workgroup");
};

// Staging registers for one key/value block, as vector values rather than
// float4 arrays: carried across the loop back-edge, the arrays were left in
// scratch memory.  Element 4f + e is component e of float4 number f.
template <int N>
using f32v = float __attribute__((ext_vector_type(N)));
template <int DP, int NT>
struct KvRegs {
  f32v<4 * SdpaCfg<DP, NT>::K_F4> k;
  f32v<16 * SdpaCfg<DP, NT>::V_PER> v;
};

// x combined with x from lane l ^ 32, the same value in both halves.
// v_permlane32_swap of (x, x) returns, per lane, {x[l & 31], x[(l & 31) + 32]}.
__device__ __forceinline__ float half_swap_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_swap_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

__device__ __forceinline__ float4 get4(const float* p) { return *reinterpret_cast<const float4*>(p); }

template <int DP, int NT, bool FULL>
__device__ __forceinline__ void load_k(const float* __restrict__ kh, long long ldk, int Skv, int D, int kb, int tid,
                                       KvRegs<DP, NT>& r) {
  using G = SdpaCfg<DP, NT>;
#pragma unroll
  for (int f = 0; f < G::K_F4; ++f) {
    const int idx0 = tid + f * NT;
    const int idx = (G::K_TOT % NT == 0 || idx0 < G::K_TOT) ? idx0 : 0;  // past the tile: reload float4 0 (unused)
    const int key = idx / G::KD4, d0 = (idx % G::KD4) * 4;
    const int gk = kb + key;
    float t[4];
    if (FULL) {
      const float4 x = get4(kh + gk * ldk + d0);
      t[0] = x.x; t[1] = x.y; t[2] = x.z; t[3] = x.w;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) t[e] = (gk < Skv && d0 + e < D) ? kh[gk * ldk + d0 + e] : 0.0f;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) r.k[4 * f + e] = t[e];
  }
}

template <int DP, int NT, bool FULL>
__device__ __forceinline__ void load_v(const float* __restrict__ vh, long long ldv, int Skv, int D, int kb, int tid,
                                       KvRegs<DP, NT>& r) {
  using G = SdpaCfg<DP, NT>;
#pragma unroll
  for (int p = 0; p < G::V_PER; ++p) {
    const int idx = tid + p * NT;
    const int blk = idx < G::V_BLK ? idx : 0;  // threads past the tile reload block 0 (unused)
    const int kq = blk / G::KD4, dq = blk % G::KD4;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int gk = kb + 4 * kq + e, d0 = 4 * dq;
      float t[4];
      if (FULL) {
        const float4 x = get4(vh + gk * ldv + d0);
        t[0] = x.x; t[1] = x.y; t[2] = x.z; t[3] = x.w;
      } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) t[c] = (gk < Skv && d0 + c < D) ? vh[gk * ldv + d0 + c] : 0.0f;
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) r.v[16 * p + 4 * e + c] = t[c];
    }
  }
}

template <int DP, int NT>
__device__ __forceinline__ void store_kv(float* __restrict__ ks, float* __restrict__ vt, int tid,
                                         const KvRegs<DP, NT>& r) {
  using G = SdpaCfg<DP, NT>;
#pragma unroll
  for (int f = 0; f < G::K_F4; ++f) {
    const int idx = tid + f * NT;
    if (G::K_TOT % NT == 0 || idx < G::K_TOT) {
      const int key = idx / G::KD4, d0 = (idx % G::KD4) * 4;
      *reinterpret_cast<float4*>(ks + key * G::KLD + d0) =
          make_float4(r.k[4 * f], r.k[4 * f + 1], r.k[4 * f + 2], r.k[4 * f + 3]);
    }
  }
#pragma unroll
  for (int p = 0; p < G::V_PER; ++p) {
    const int idx = tid + p * NT;
    if (G::V_BLK % NT == 0 || idx < G::V_BLK) {
      // transpose the 4(key) x 4(d) block: row d of Vt gets keys 4kq .. 4kq + 3
      const int kq = idx / G::KD4, dq = idx % G::KD4;
      float* base = vt + (4 * dq) * kVLD + 4 * kq;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        *reinterpret_cast<float4*>(base + c * kVLD) =
            make_float4(r.v[16 * p + c], r.v[16 * p + 4 + c], r.v[16 * p + 8 + c], r.v[16 * p + 12 + c]);
    }
  }
}

// ---- D <= 128 ----
// LDS of one key block, three parts each of K, [d octet][32 keys][8 d], and of V, [4 key octets]
// [DP][8 keys].  K's keys are permuted by the octet (key ^ octet % 8), so that the eight lanes of
// a store phase, eight octets of one key, cover different banks.  At D = 128 the smallest part
// of q for QL of the eight 16-d steps is kept in LDS too: with all 96 registers of q's parts
// resident the kernel spilled (57 registers; two wavefronts per SIMD leave 256).
template <int DP, int NW>
struct FwdCfg {
  static constexpr int NT = 64 * NW, BQ = 32 * NW;
  static constexpr int NO = DP / 8;                    // d octets
  static constexpr int KSTR = kBKV * 16, VSTR = DP * 16;
  static constexpr int KBYTES = 3 * NO * KSTR, VBYTES = 3 * 4 * VSTR;
  static constexpr int QL = DP == 128 ? 7 : 0;
  static constexpr int NCH = kBKV * NO;                // octets of K, and of V, per block
  static constexpr int CH = (NCH + NT - 1) / NT;       // per thread
  static_assert(2 * (KBYTES + VBYTES) + QL * NT * 16 <= 160 * 1024 - 16, "LDS");
};

// DF: D == DP; RAG: Skv % 32 != 0.  splits > 1: split blockIdx.y of the keys, unnormalised
// results to part.
template <int DP, int NW, bool DF, bool RAG>
__global__ __launch_bounds__(64 * NW) void sdpa_fwd_kernel(
    int H, int group, int BH, int Sq, int Skv, int D, float qscale, int causal, const float* __restrict__ q,
    const float* __restrict__ k, const float* __restrict__ v, float* __restrict__ o, bch::SdpaStrides st,
    int qblocks, float* __restrict__ part) {
  using G = FwdCfg<DP, NW>;
  constexpr int NT = G::NT, NO = G::NO, NC = DP / 16, NBK = DP / 32;
  __shared__ __attribute__((aligned(16))) char k_lds[2 * G::KBYTES], v_lds[2 * G::VBYTES];
  __shared__ u32x4 q_lds[G::QL > 0 ? G::QL * NT : 1];
  __shared__ int big_seen;

  // causal: query-block major, all heads' longest query blocks first.
  // non-causal: head-major over an XCD-contiguous remap of the grid.
  int qi, bh;
  if (causal) {
    qi = blockIdx.x / BH;
    bh = blockIdx.x % BH;
  } else {
    const int nb = gridDim.x;
    int L = blockIdx.x;
    if ((nb & 7) == 0) L = (L & 7) * (nb >> 3) + (L >> 3);
    bh = L / qblocks;
    qi = L - bh * qblocks;
  }
  const int qb = causal ? qblocks - 1 - qi : qi;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, lh = lane >> 5;
  const int q0w = qb * G::BQ + wave * 32;  // first query of this wavefront
  const int myq = q0w + li;

  const int bi = bh / H, hq = bh - bi * H, hk = hq / group;
  const float* kh = k + bi * st.k.batch + hk * st.k.head;
  const float* vh = v + bi * st.v.batch + hk * st.v.head;
  float* oh = o + bi * st.o.batch + hq * st.o.head;
  // queries past the end repeat the last one and are not stored
  const float* qr = q + bi * st.q.batch + hq * st.q.head + (long long)min(myq, Sq - 1) * st.q.row;

  if (tid == 0) big_seen = 0;

  // eight floats of a row from column d0 on, zeros from D on
  auto row8 = [&](const float* row, int d0, float (&x)[8]) {
    if (DF) {
      typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
      const f32x4u a = *reinterpret_cast<const f32x4u*>(row + d0), b = *reinterpret_cast<const f32x4u*>(row + d0 + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = a[e];
        x[4 + e] = b[e];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float t = row[min(d0 + e, D - 1)];
        x[e] = d0 + e < D ? t : 0.0f;
      }
    }
  };

  // ---- q parts: step c holds q[myq][16c + 8lh .. +7] * scale * log2(e) ----
  u32x4 qf[NC][3];
  float mq = 0.0f;  // largest magnitude
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    float x[8];
    row8(qr, 16 * c + 8 * lh, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) mq = fmaxf(mq, fabsf(x[e] * qscale));
    split8(x, qf[c], qscale * bch::kSplitScale);
    if (c < G::QL) q_lds[c * NT + tid] = qf[c][2];  // read back by this lane alone
  }
  const bool q_big = __any(mq >= kScoreBig);  // settled here: later, the floats of q would stay in registers

  f32x16 oacc[NBK];
  float m_ref, l_run;
  auto reset = [&]() {
#pragma unroll
    for (int b = 0; b < NBK; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[b][r] = 0.0f;
    m_ref = -INFINITY;
    l_run = 0.0f;
  };
  reset();

  // this workgroup's key blocks
  const int kend = causal ? min(Skv, qb * G::BQ + G::BQ) : Skv;
  const int nall = (kend + kBKV - 1) / kBKV;
  const int t0 = (int)((long long)nall * blockIdx.y / gridDim.y);
  const int t1 = (int)((long long)nall * (blockIdx.y + 1) / gridDim.y);

  // ---- global -> registers -> parts in LDS ----
  // octet ch of K: key ch / NO, d 8 (ch % NO) .. +7; of V: column ch % DP, key octet ch / DP (keys
  // 16 (oct / 2) + 4 (oct % 2) + {0..3, 8..11}).  Keys past the end repeat the last one; their
  // scores are masked and their V rows zeroed.
  float rk[G::CH][8], rv[G::CH][8];
  float mk = 0.0f;  // largest magnitude of the K that this thread has split
  auto load_k = [&](int t) {
#pragma unroll
    for (int c = 0; c < G::CH; ++c) {
      const int ch = (G::NCH % NT == 0) ? tid + c * NT : min(tid + c * NT, G::NCH - 1);
      const int key = t * kBKV + ch / NO;
      row8(kh + (long long)(RAG ? min(key, Skv - 1) : key) * st.k.row, 8 * (ch % NO), rk[c]);
    }
  };
  auto load_v = [&](int t) {
#pragma unroll
    for (int c = 0; c < G::CH; ++c) {
      const int ch = (G::NCH % NT == 0) ? tid + c * NT : min(tid + c * NT, G::NCH - 1);
      // one key octet for a whole wavefront where DP allows: scalar row addresses
      const int oct = DP % 64 == 0 ? __builtin_amdgcn_readfirstlane(ch / DP) : ch / DP;
      const unsigned d = DF ? ch % DP : min(ch % DP, D - 1);
      const int key0 = t * kBKV + 16 * (oct >> 1) + 4 * (oct & 1);
      const float* v0r = vh + (long long)key0 * st.v.row;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int dk = (e & 3) + 8 * (e >> 2);
        rv[c][e] = (RAG ? vh + (long long)min(key0 + dk, Skv - 1) * st.v.row : v0r + dk * st.v.row)[d];
      }
    }
  };
  auto zero_tail = [&](int t) {  // V rows past the last key
#pragma unroll
    for (int c = 0; c < G::CH; ++c) {
      const int oct = (tid + c * NT) / DP, key0 = t * kBKV + 16 * (oct >> 1) + 4 * (oct & 1);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (key0 + (e & 3) + 8 * (e >> 2) >= Skv) rv[c][e] = 0.0f;
    }
  };
  u32x4 kp[G::CH][3], vp[G::CH][3];
  // one of the 8 CH pairs of floats of this thread's octets: V's first, then K's
  constexpr int UNITS = 8 * G::CH;
  auto split_unit = [&](int u) {
    const int c = (u >> 2) % G::CH, e = u & 3;
    float& x = u < UNITS / 2 ? rv[c][2 * e] : rk[c][2 * e];
    float& y = u < UNITS / 2 ? rv[c][2 * e + 1] : rk[c][2 * e + 1];
    if (u >= UNITS / 2) mk = fmaxf(mk, fmaxf(fabsf(x), fabsf(y)));
    x *= bch::kSplitScale;
    y *= bch::kSplitScale;
    bch::split2(x, y, u < UNITS / 2 ? vp[c] : kp[c], e);
  };
  auto store_k = [&](int buf) {
    char* s = k_lds + buf * G::KBYTES;
#pragma unroll
    for (int c = 0; c < G::CH; ++c) {
      const int ch = tid + c * NT;
      if (G::NCH % NT == 0 || ch < G::NCH) {
#pragma unroll
        for (int p3 = 0; p3 < 3; ++p3)
          *reinterpret_cast<u32x4*>(s + (p3 * NO + ch % NO) * G::KSTR + ((ch / NO) ^ (ch % NO & 7)) * 16) = kp[c][p3];
      }
    }
  };
  auto store_v = [&](int buf) {
    char* s = v_lds + buf * G::VBYTES;
#pragma unroll
    for (int c = 0; c < G::CH; ++c) {
      const int ch = tid + c * NT;
      if (G::NCH % NT == 0 || ch < G::NCH) {
#pragma unroll
        for (int p3 = 0; p3 < 3; ++p3)
          *reinterpret_cast<u32x4*>(s + (p3 * 4 + ch / DP) * G::VSTR + (ch % DP) * 16) = vp[c][p3];
      }
    }
  };

  // value r of a score block: key kb + 8(r/4) + 4lh + r%4, query myq
  auto mask = [&](f32x16& s, int kb) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = kb + 8 * (r >> 2) + 4 * lh + (r & 3);
      if (key >= Skv || (causal && key > myq)) s[r] = -INFINITY;
    }
  };
  // Scores -> probabilities against the reference max, which moves when a block exceeds it by
  // more than 2^kLazy, and their parts pf, in kPieces pieces that a caller may set between MFMAs.
  // unit: the scores' scale.  (A reference 16 lower would scale the probabilities for nothing, but
  // larger exponents round more: error at the timed shape 3.8e-7 -> 4.4e-7.)
  // alpha: what the results so far are to be multiplied by (rescale).
  u32x4 pf[2][3];  // parts of the last block's probabilities
  float bm, m_use, rs, alpha;
  constexpr int kPieces = 20;
  auto piece = [&](float unit, f32x16& s, int i) {
    if (i == 0) {
      bm = s[0];
#pragma unroll
      for (int r = 1; r < 8; ++r) bm = fmaxf(bm, s[r]);
    } else if (i == 1) {
#pragma unroll
      for (int r = 8; r < 16; ++r) bm = fmaxf(bm, s[r]);
      bm = half_swap_max(bm) * unit;
    } else if (i == 2) {
      const bool move = bm > m_ref + kLazy;  // -inf reference: any finite block max moves it
      const float m_new = move ? bm : m_ref;
      alpha = move ? (m_ref == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_ref - m_new)) : 1.0f;
      m_ref = m_new;
      m_use = (m_ref == -INFINITY) ? 0.0f : m_ref;
      rs = 0.0f;
    } else if (i < 11) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int r = 2 * (i - 3) + e;
        s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], unit, -m_use));
        rs += s[r];
      }
    } else if (i == 11) {
      l_run = l_run * alpha + half_swap_sum(rs);
    } else {
      const int u = i - 12, h = u >> 2, e = u & 3;
      float x = s[8 * h + 2 * e] * bch::kSplitScale, y = s[8 * h + 2 * e + 1] * bch::kSplitScale;
      bch::split2(x, y, pf[h], e);
    }
  };
  auto softmax = [&](float unit, f32x16& s) {  // without the parts
#pragma unroll
    for (int i = 0; i < 12; ++i) piece(unit, s, i);
    return alpha;
  };
  auto rescale = [&](float alpha) {
    if (__any(alpha != 1.0f)) {
#pragma unroll
      for (int b = 0; b < NBK; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[b][r] *= alpha;
    }
  };

  // the scores of the block in buffer buf, with work(i) behind MFMA i of 6 NC
  auto qk = [&](int buf, f32x16& s, auto&& work) {
    const char* ks = k_lds + buf * G::KBYTES + lh * G::KSTR;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.0f;
    u32x4 kf[2][3], q2[2];
    auto read = [&](int c) {  // octet 2c + lh
      const int key = li ^ ((2 * c + lh) & 7);
#pragma unroll
      for (int p3 = 0; p3 < 3; ++p3)
        kf[c & 1][p3] = *reinterpret_cast<const u32x4*>(ks + (p3 * NO + 2 * c) * G::KSTR + key * 16);
      q2[c & 1] = c < G::QL ? q_lds[c * NT + tid] : qf[c][2];
    };
    read(0);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (c + 1 < NC) read(c + 1);
#pragma unroll
      for (int x = 0; x < 6; ++x) {
        const int pb = bch::kPartB[x];
        s = bf16_mm(kf[c & 1][bch::kPartA[x]], pb == 2 ? q2[c & 1] : qf[c][pb], s);
        work(6 * c + x);
      }
    }
  };
  // O += V^T P^T of the block in buffer buf
  auto pv = [&](int buf) {
    const char* vs = v_lds + buf * G::VBYTES + lh * G::VSTR + li * 16;
    u32x4 vf[2][3];
    auto read = [&](int i) {  // 16-k step i / NBK, O block i % NBK
#pragma unroll
      for (int p3 = 0; p3 < 3; ++p3)
        vf[i & 1][p3] = *reinterpret_cast<const u32x4*>(vs + (p3 * 4 + 2 * (i / NBK)) * G::VSTR + (i % NBK) * 512);
    };
    read(0);
#pragma unroll
    for (int i = 0; i < 2 * NBK; ++i) {
      if (i + 1 < 2 * NBK) read(i + 1);
#pragma unroll
      for (int y = 0; y < 6; ++y)
        oacc[i % NBK] = bf16_mm(vf[i & 1][bch::kPartA[y]], pf[i / NBK][bch::kPartB[y]], oacc[i % NBK]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // Block t's scores run over the conversion of block t + 1's K and V (stored to the other buffers,
  // which the previous barrier released), a few VALU operations behind each MFMA (pinned there by
  // scheduling barriers, which also keep the reads of LDS from piling up registers); then the
  // softmax and the PV product, under which the SIMD's other wavefront has its turn.  Blocks past
  // the end are clamped to the last one (reloaded, never read).  Measured against one wavefront per
  // SIMD (128 queries, block t - 1's PV product set between block t's softmax operations): 880 ->
  // 707 us (B 4, H 32, S 2048, D 128, causal).
  auto stage = [&](int t) {  // block t + 1 to the other buffers, block t + 2's loads
    const int nxt = (t - t0 + 1) & 1;
    store_v(nxt);
    store_k(nxt);
    load_k(min(t + 2, t1 - 1));
    load_v(min(t + 2, t1 - 1));
  };
  auto iteration = [&](auto masked, int t) {
    const int cur = (t - t0) & 1;
    constexpr int NQ = 6 * NC;
    if (decltype(masked)::value && RAG && min(t + 1, t1 - 1) * kBKV + kBKV > Skv) zero_tail(min(t + 1, t1 - 1));
    f32x16 s;
    qk(cur, s, [&](int i) {
#pragma unroll
      for (int u = 0; u < UNITS; ++u)
        if (u * NQ / UNITS == i) split_unit(u);
      __builtin_amdgcn_sched_barrier(0);
    });
    stage(t);
    __builtin_amdgcn_sched_barrier(0);
    if (decltype(masked)::value) mask(s, t * kBKV);
    rescale(softmax(bch::kSplitUnscale, s));
#pragma unroll
    for (int i = 12; i < kPieces; ++i) piece(bch::kSplitUnscale, s, i);
    __builtin_amdgcn_sched_barrier(0);
    pv(cur);
    __syncthreads();
  };
  // the first block past this wavefront's last query (it still stages K and V from there on), and
  // the first one with keys to mask or whose next block has V rows to zero
  const int tw = q0w >= Sq ? t0 : causal ? max(t0, min(t1, (q0w + 31) / kBKV + 1)) : t1;
  const int tm = min(tw, min(causal ? q0w / kBKV : t1, RAG ? Skv / kBKV - 1 : t1));
  if (t0 < t1) {
    load_k(t0);
    load_v(t0);
    if (RAG && t0 * kBKV + kBKV > Skv) zero_tail(t0);
#pragma unroll
    for (int u = 0; u < UNITS; ++u) split_unit(u);
    store_v(0);
    store_k(0);
    load_k(min(t0 + 1, t1 - 1));
    load_v(min(t0 + 1, t1 - 1));
  }
  __syncthreads();
  int t = t0;
#pragma unroll 1
  for (; t < tm; ++t) iteration(std::false_type{}, t);
#pragma unroll 1
  for (; t < tw; ++t) iteration(std::true_type{}, t);
#pragma unroll 1
  for (; t < t1; ++t) {
    if (RAG && min(t + 1, t1 - 1) * kBKV + kBKV > Skv) zero_tail(min(t + 1, t1 - 1));
#pragma unroll
    for (int u = 0; u < UNITS; ++u) split_unit(u);
    stage(t);
    __syncthreads();
  }

  // ---- O scaled back; where the parts cannot stand for the operands, these queries again in f32 ----
  bool redo;
  {
    float z = l_run * 0.0f;
#pragma unroll
    for (int b = 0; b < NBK; ++b) {
      oacc[b] *= bch::kSplitUnscale;
#pragma unroll
      for (int r = 0; r < 16; ++r) z = fmaf(oacc[b][r], 0.0f, z);
    }
    if (mk >= kScoreBig) big_seen = 1;
    __syncthreads();
    redo = q_big || big_seen != 0 || __any(z != 0.0f);
  }
  if (redo && q0w < Sq) {
    // 16 d of a block's K and q, then its V, are loaded before their MFMAs (step e contracts d 16c + e
    // and 16c + 8 + e).  Ends once every query's sum is NaN.  Measured (us, one box, B 4, H 32, S 2048,
    // D 128, causal; a kernel on the f32 instruction throughout / an element loaded, then
    // multiplied, at a time / this): an infinite V in every head 1095 / 4945 / 2298, in one head
    // 1094 / 2250 / 1095, a NaN key in every head 1091 / 4918 / 711.  (With all of K and q loaded at
    // once 2050, but the loop above then ran 3% slower, with its instructions the same.)
    reset();
#pragma unroll 1
    for (int t = t0; t < t1; ++t) {
      const int kb = t * kBKV;
      if (causal && kb > q0w + 31) break;
      const float* const kr = kh + (long long)min(kb + li, Skv - 1) * st.k.row;
      f32x16 s;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = 0.0f;
#pragma unroll 1
      for (int d0 = 0; d0 < D; d0 += 16) {
        float x[8], y[8];
        row8(kr, d0 + 8 * lh, x);
        row8(qr, d0 + 8 * lh, y);
#pragma unroll
        for (int e = 0; e < 8; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], y[e] * qscale, s, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      float vx[16][NBK];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = kb + 8 * (r >> 2) + 4 * lh + (r & 3);
        const float* const vr = vh + (long long)min(key, Skv - 1) * st.v.row;
#pragma unroll
        for (int b = 0; b < NBK; ++b) vx[r][b] = vr[min(32 * b + li, D - 1)];
      }
      __builtin_amdgcn_sched_barrier(0);
      if (kb + kBKV > Skv || (causal && kb + kBKV - 1 > q0w)) mask(s, kb);
      rescale(softmax(1.0f, s));
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const bool in = kb + 8 * (r >> 2) + 4 * lh + (r & 3) < Skv;
#pragma unroll
        for (int b = 0; b < NBK; ++b)
          oacc[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(in ? vx[r][b] : 0.0f, s[r], oacc[b], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (__all(l_run != l_run)) break;
    }
  }

  // ---- epilogue: value r of block b is d = 32b + 8(r/4) + 4lh + r%4 ----
  if (myq < Sq) {
    float inv = 1.0f;
    float* dst = oh + (long long)myq * st.o.row;
    if (gridDim.y > 1) {
      float* p = part + ((long long)bh * gridDim.y + blockIdx.y) * bch::sdpa_part_floats(Sq, D);
      dst = p + (long long)myq * D;
      if (lh == 0) {
        p[(long long)Sq * D + 2 * myq] = m_ref;
        p[(long long)Sq * D + 2 * myq + 1] = l_run;
      }
    } else {
      inv = 1.0f / l_run;
    }
#pragma unroll
    for (int b = 0; b < NBK; ++b) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int d = 32 * b + 8 * (r >> 2) + 4 * lh + (r & 3);
        if (DF || d < D) dst[d] = oacc[b][r] * inv;
      }
    }
  }
}

// ---- 128 < D <= 256: v_mfma_f32_16x16x4_f32, 16 queries per wavefront ----
// The 32x32 layout above keeps D/2 floats of q and D/2 of O per lane: at
// D = 256 that is 256 registers before staging and scores, one wavefront per
// SIMD, with the softmax of each block exposed on its SIMD.  Here a
// wavefront owns 16 queries, so q and O take D/4 floats each (64 + 64 at
// D = 256) and two wavefronts share each SIMD: 8 wavefronts = 128 queries
// per workgroup, the same K/V tile reuse and LDS layout as the 32x32 kernel
// (one workgroup per CU at 137 KB of LDS for D = 256).
//   S^T = K Q^T on 16 x 16 blocks: lane (g = l / 16, i = l % 16) supplies
//     K[key 16 sb + i][d] and q[query i][d] with d = 16 c + 4 g + e in step
//     (c, e), so one 128-bit LDS read of K and one register float4 of q feed
//     four MFMAs; value r of the result is key 16 sb + 4 g + r of query i.
//     A 32-key block is two such chains (sb = 0, 1): 8 scores per lane.
//   Row max and sum: in-lane over the 8, then across the four lanes
//     i, i + 16, i + 32, i + 48 of a query (v_permlane16_swap then
//     v_permlane32_swap; every lane of a query gets the same bits).
//   O^T += V^T P^T: step (sb, r) contracts key 16 sb + 4 g + r, whose P is
//     this lane's score r of chain sb; V^T comes from the transposed V tile
//     as one 128-bit read per four MFMAs.  Value r of O block db is
//     d = 16 db + 4 g + r of query i: the epilogue stores a float4.
// The online softmax (lazy reference max), causal skipping and masking and
// the workgroup order are those of sdpa_fwd_kernel.
// Measured at B=4, H=32, S=2048, D=256 (one box): 4.27 / 2.27 ms non-causal /
// causal (81.9% / 77.1% of FP32 MFMA peak), against 5.01 / 2.75 ms for
// sdpa_fwd_kernel at D = 256 (one wavefront per SIMD, accumulators in
// AGPRs).  D = 160 / 192 / 224: 75% / 77% / 79% non-causal.  For D <= 128
// this layout is slower than the 32x32 kernel (2.15 against 2.05 ms at
// config 5, 4 wavefronts per SIMD), so it starts above 128.
constexpr int kNT16 = 512;        // threads per workgroup: 8 wavefronts
constexpr int kBQ16 = kNT16 / 4;  // queries per workgroup (16 per wavefront)

typedef float f32x4v __attribute__((ext_vector_type(4)));

// x combined over the lanes l, l ^ 16, l ^ 32, l ^ 48 (the four lanes of one
// query), the same bits in all four: v_permlane16_swap of (x, x) returns
// {x[l & ~16], x[l | 16]} and v_permlane32_swap {x[l & ~32], x[l | 32]}.
__device__ __forceinline__ float quad_swap_max(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float quad_swap_sum(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <int DP, bool FULL>
__global__ __launch_bounds__(kNT16, 2) void sdpa_fwd16_kernel(
    int H, int group, int BH, int Sq, int Skv, int D, float qscale, int causal, const float* __restrict__ q,
    const float* __restrict__ k, const float* __restrict__ v, float* __restrict__ o, bch::SdpaStrides st,
    int qblocks) {
  using G = SdpaCfg<DP, kNT16>;
  constexpr int KLD = G::KLD, NT = kNT16;
  extern __shared__ float4 smem4[];
  float* smem = reinterpret_cast<float*>(smem4);
  float* Ks = smem;                        // [2][kBKV][KLD]
  float* Vt = smem + 2 * kBKV * KLD;       // [2][DP][kVLD]

  int qi, bh;
  if (causal) {
    qi = blockIdx.x / BH;
    bh = blockIdx.x % BH;
  } else {
    const int nb = gridDim.x;
    int L = blockIdx.x;
    if ((nb & 7) == 0) L = (L & 7) * (nb >> 3) + (L >> 3);
    bh = L / qblocks;
    qi = L - bh * qblocks;
  }
  const int qb = causal ? qblocks - 1 - qi : qi;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int q0w = qb * kBQ16 + wave * 16;  // first query of this wavefront
  const int myq = q0w + li;

  const int bi = bh / H, hq = bh - bi * H, hk = hq / group;
  const float* qh = q + bi * st.q.batch + hq * st.q.head;
  const float* kh = k + bi * st.k.batch + hk * st.k.head;
  const float* vh = v + bi * st.v.batch + hk * st.v.head;
  float* oh = o + bi * st.o.batch + hq * st.o.head;

  // ---- q operand: qf[c] = q[myq][16c + 4lg .. +3] * scale * log2(e) ----
  float4 qf[DP / 16];
#pragma unroll
  for (int c = 0; c < DP / 16; ++c) {
    const int d0 = 16 * c + 4 * lg;
    float t[4];
    if (FULL) {
      const float4 x = *reinterpret_cast<const float4*>(qh + myq * st.q.row + d0);
      t[0] = x.x; t[1] = x.y; t[2] = x.z; t[3] = x.w;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) t[e] = (myq < Sq && d0 + e < D) ? qh[myq * st.q.row + d0 + e] : 0.0f;
    }
    qf[c] = make_float4(t[0] * qscale, t[1] * qscale, t[2] * qscale, t[3] * qscale);
  }

  f32x4v oacc[DP / 16];
#pragma unroll
  for (int b = 0; b < DP / 16; ++b) oacc[b] = (f32x4v){0.f, 0.f, 0.f, 0.f};
  float m_ref = -INFINITY, l_run = 0.0f;

  int kend = Skv;
  if (causal) kend = min(Skv, qb * kBQ16 + kBQ16);
  const int nkb = (kend + kBKV - 1) / kBKV;

  KvRegs<DP, NT> kv;
  load_k<DP, NT, FULL>(kh, st.k.row, Skv, D, 0, tid, kv);
  load_v<DP, NT, FULL>(vh, st.v.row, Skv, D, 0, tid, kv);
  store_kv<DP, NT>(Ks, Vt, tid, kv);
  load_k<DP, NT, FULL>(kh, st.k.row, Skv, D, min(1, nkb - 1) * kBKV, tid, kv);
  load_v<DP, NT, FULL>(vh, st.v.row, Skv, D, min(1, nkb - 1) * kBKV, tid, kv);
  __syncthreads();

  for (int t = 0; t < nkb; ++t) {
    const int cur = t & 1;
    const int kb = t * kBKV;
    store_kv<DP, NT>(Ks + (cur ^ 1) * kBKV * KLD, Vt + (cur ^ 1) * DP * kVLD, tid, kv);
    const int kbn = min(t + 2, nkb - 1) * kBKV;
    load_k<DP, NT, FULL>(kh, st.k.row, Skv, D, kbn, tid, kv);
    load_v<DP, NT, FULL>(vh, st.v.row, Skv, D, kbn, tid, kv);

    const bool active = (q0w < Sq) && !(causal && kb > q0w + 15);
    if (active) {
      const float* ks = Ks + cur * kBKV * KLD + li * KLD + 4 * lg;
      f32x4v s[2];
      s[0] = s[1] = (f32x4v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < DP / 16; ++c) {
#pragma unroll
        for (int sb = 0; sb < 2; ++sb) {
          const float4 kf = *reinterpret_cast<const float4*>(ks + sb * 16 * KLD + 16 * c);
          s[sb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf.x, qf[c].x, s[sb], 0, 0, 0);
          s[sb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf.y, qf[c].y, s[sb], 0, 0, 0);
          s[sb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf.z, qf[c].z, s[sb], 0, 0, 0);
          s[sb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf.w, qf[c].w, s[sb], 0, 0, 0);
        }
      }
      // value r of chain sb: key kb + 16 sb + 4 lg + r, query myq
      const bool need_mask = (!FULL && kb + kBKV > Skv) || (causal && kb + kBKV - 1 > q0w);
      if (need_mask) {
#pragma unroll
        for (int sb = 0; sb < 2; ++sb)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int key = kb + 16 * sb + 4 * lg + r;
            if (key >= Skv || (causal && key > myq)) s[sb][r] = -INFINITY;
          }
      }
      float bm = s[0][0];
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
#pragma unroll
        for (int r = 0; r < 4; ++r) bm = fmaxf(bm, s[sb][r]);
      bm = quad_swap_max(bm);
      const bool move = bm > m_ref + kLazy;
      if (__any(move)) {
        const float m_new = move ? bm : m_ref;
        const float alpha = (m_ref == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(m_ref - m_new);
        l_run *= alpha;
#pragma unroll
        for (int b = 0; b < DP / 16; ++b) oacc[b] *= alpha;
        m_ref = m_new;
      }
      const float m_use = (m_ref == -INFINITY) ? 0.0f : m_ref;
      float rs = 0.0f;
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[sb][r] = __builtin_amdgcn_exp2f(s[sb][r] - m_use);
          rs += s[sb][r];
        }
      rs = quad_swap_sum(rs);
      l_run += rs;

      const float* vs = Vt + cur * DP * kVLD + li * kVLD + 4 * lg;
#pragma unroll
      for (int db = 0; db < DP / 16; ++db) {
#pragma unroll
        for (int sb = 0; sb < 2; ++sb) {
          const float4 vf = *reinterpret_cast<const float4*>(vs + db * 16 * kVLD + 16 * sb);
          oacc[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf.x, s[sb][0], oacc[db], 0, 0, 0);
          oacc[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf.y, s[sb][1], oacc[db], 0, 0, 0);
          oacc[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf.z, s[sb][2], oacc[db], 0, 0, 0);
          oacc[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf.w, s[sb][3], oacc[db], 0, 0, 0);
        }
      }
    }
    __syncthreads();
  }

  // ---- epilogue: value r of block db is d = 16 db + 4 lg + r ----
  if (myq < Sq) {
    const float inv = 1.0f / l_run;
#pragma unroll
    for (int db = 0; db < DP / 16; ++db) {
      const int d0 = 16 * db + 4 * lg;
      if (FULL) {
        *reinterpret_cast<float4*>(oh + myq * st.o.row + d0) =
            make_float4(oacc[db][0] * inv, oacc[db][1] * inv, oacc[db][2] * inv, oacc[db][3] * inv);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (d0 + r < D) oh[myq * st.o.row + d0 + r] = oacc[db][r] * inv;
      }
    }
  }
}

template <int DP, bool FULL>
hipError_t launch_dp16(hipStream_t s, int B, int H, int Hkv, int Sq, int Skv, int D, float scale, int causal,
                       const float* q, const float* k, const float* v, float* o, const bch::SdpaStrides& st) {
  using G = SdpaCfg<DP, kNT16>;
  const int qblocks = (Sq + kBQ16 - 1) / kBQ16;
  const long long blocks = (long long)B * H * qblocks;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  const size_t lds = sizeof(float) * G::LDS_FLOATS;
  auto kern = sdpa_fwd16_kernel<DP, FULL>;
  hipError_t e = bch::ensure_dynamic_lds(reinterpret_cast<const void*>(kern), (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kNT16), lds, s, H, H / Hkv, B * H, Sq, Skv, D,
                     scale * kLog2E, causal, q, k, v, o, st, qblocks);
  return hipGetLastError();
}

template <int DP, int NW, bool DF, bool RAG>
hipError_t launch_dp(hipStream_t s, int B, int H, int Hkv, int Sq, int Skv, int D, float scale, int causal,
                     const float* q, const float* k, const float* v, float* o, const bch::SdpaStrides& st, int splits,
                     float* part) {
  using G = FwdCfg<DP, NW>;
  const int qblocks = (Sq + G::BQ - 1) / G::BQ;
  const long long blocks = (long long)B * H * qblocks;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  auto kern = sdpa_fwd_kernel<DP, NW, DF, RAG>;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks, splits), dim3(G::NT), 0, s, H, H / Hkv, B * H, Sq, Skv, D,
                     scale * kLog2E, causal, q, k, v, o, st, qblocks, part);
  return hipGetLastError();
}

// 256-query workgroups where they give every CU one; else 128-query ones, with the keys split
// until the CUs are filled or a split is down to two key blocks.
struct FwdPlan {
  int nw = 8, splits = 1;
};
FwdPlan fwd_plan(int B, int H, int Sq, int Skv) {
  FwdPlan p;
  const long long cu = bch::device_cu_count(), bh = (long long)B * H;
  if (bh * ((Sq + 255) / 256) >= cu) return p;
  p.nw = 4;
  const long long blocks = bh * ((Sq + 127) / 128);
  p.splits = (int)std::max(1LL, std::min<long long>({cu / blocks, (Skv + 63) / 64, 16}));
  return p;
}

bool aligned16(const float* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
bool mult4(const bch::SdpaLayout& l) { return l.batch % 4 == 0 && l.head % 4 == 0 && l.row % 4 == 0; }

template <int DP>
hipError_t launch_d(hipStream_t s, int B, int H, int Hkv, int Sq, int Skv, int D, float scale, int causal,
                    const float* q, const float* k, const float* v, float* o, const bch::SdpaStrides& st,
                    const FwdPlan& p, float* part) {
#define BCH_FWD(NW_, DF_, RAG_) \
  launch_dp<DP, NW_, DF_, RAG_>(s, B, H, Hkv, Sq, Skv, D, scale, causal, q, k, v, o, st, p.splits, part)
#define BCH_FWD_NW(NW_)                                                     \
  (D == DP ? (rag ? BCH_FWD(NW_, true, true) : BCH_FWD(NW_, true, false)) \
           : (rag ? BCH_FWD(NW_, false, true) : BCH_FWD(NW_, false, false)))
  const bool rag = Skv % kBKV != 0;
  return p.nw == 8 ? BCH_FWD_NW(8) : BCH_FWD_NW(4);
#undef BCH_FWD_NW
#undef BCH_FWD
}

// 128 < D <= 256: the 16-query-per-wavefront kernel
template <int DP>
hipError_t launch_d16(hipStream_t s, int B, int H, int Hkv, int Sq, int Skv, int D, float scale, int causal,
                      const float* q, const float* k, const float* v, float* o, const bch::SdpaStrides& st) {
  const bool full = D == DP && Sq % kBQ16 == 0 && Skv % kBKV == 0 && aligned16(q) && aligned16(k) && aligned16(v) &&
                    aligned16(o) && mult4(st.q) && mult4(st.k) && mult4(st.v) && mult4(st.o);
  if (full) return launch_dp16<DP, true>(s, B, H, Hkv, Sq, Skv, D, scale, causal, q, k, v, o, st);
  return launch_dp16<DP, false>(s, B, H, Hkv, Sq, Skv, D, scale, causal, q, k, v, o, st);
}

}  // namespace

namespace bch {

size_t sdpa_fwd_workspace_bytes(int B, int H, int Sq, int Skv, int D) {
  if (D > 128) return 0;
  const FwdPlan p = fwd_plan(B, H, Sq, Skv);
  return p.splits > 1 ? sizeof(float) * (size_t)B * H * p.splits * sdpa_part_floats(Sq, D) : 0;
}

hipError_t launch_sdpa_strided(hipStream_t s, int B, int H, int Hkv, int Sq, int Skv, int D, float scale,
                               int causal, const float* q, const float* k, const float* v, float* o,
                               const SdpaStrides& st, void* ws, size_t ws_bytes) {
  if (Hkv < 1 || H % Hkv != 0) return hipErrorInvalidValue;
  if (D <= 128) {
    FwdPlan p = fwd_plan(B, H, Sq, Skv);
    if (ws_bytes < sdpa_fwd_workspace_bytes(B, H, Sq, Skv, D)) p.splits = 1;
    float* part = static_cast<float*>(ws);
    hipError_t e = D <= 32   ? launch_d<32>(s, B, H, Hkv, Sq, Skv, D, scale, causal, q, k, v, o, st, p, part)
                   : D <= 64 ? launch_d<64>(s, B, H, Hkv, Sq, Skv, D, scale, causal, q, k, v, o, st, p, part)
                   : D <= 96 ? launch_d<96>(s, B, H, Hkv, Sq, Skv, D, scale, causal, q, k, v, o, st, p, part)
                             : launch_d<128>(s, B, H, Hkv, Sq, Skv, D, scale, causal, q, k, v, o, st, p, part);
    if (e != hipSuccess || p.splits == 1) return e;
    return launch_sdpa_combine(s, B, H, H, Sq, D, p.splits, part, o, st.o);
  }
  if (D <= 160) return launch_d16<160>(s, B, H, Hkv, Sq, Skv, D, scale, causal, q, k, v, o, st);
  if (D <= 192) return launch_d16<192>(s, B, H, Hkv, Sq, Skv, D, scale, causal, q, k, v, o, st);
  if (D <= 224) return launch_d16<224>(s, B, H, Hkv, Sq, Skv, D, scale, causal, q, k, v, o, st);
  if (D <= 256) return launch_d16<256>(s, B, H, Hkv, Sq, Skv, D, scale, causal, q, k, v, o, st);
  return hipErrorInvalidValue;
}

}  // namespace bch

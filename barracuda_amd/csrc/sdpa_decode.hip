// sdpa_decode.hip -- attention forward for few query rows over many keys (a
// decode step), split over the keys.
//
// Replaces the same reference ops as sdpa_fwd.hip for calls whose query
// rows cannot fill its 128-query workgroups: one or a few query rows per
// sequence against a cache of Skv keys (ops/attention/compute.rs:21-111 with
// Sq < Skv; ops/grouped_query_attention/compute.rs:27-121 with its query
// heads sharing a key/value head).  Non-causal, D <= 128.
//
// What bounds it: reading K and V once.  A 128-query workgroup per query head
// pads 127 of its rows, reads a key/value head once per query head that
// shares it, and B * H of them need not fill the chip (8 x 32 heads, 8 key/value
// heads, one query over 4096 keys of 128: 694 us for 268 MB).  Here:
//   * Rows: the H / Hkv query heads of a key/value head and their Sq rows
//     are one list of rows, taken 16 at a time (row r: query head
//     hk * group + r / Sq, query r % Sq), so K and V are read once for all of
//     them.
//   * Keys are split over workgroups until two workgroups of four wavefronts
//     run per CU, and over the wavefronts of a workgroup in blocks of 16.
//     A wavefront needs no other: K and V go from global memory straight
//     into operand registers (v_mfma_f32_16x16x4_f32, whose k index each
//     lane group may choose), the next block's loads always in flight, with
//     no LDS and no barrier until the end.  The matrix cores could take
//     19 TB/s of K and V this way.
//   * S^T = K Q^T: lane (g = l / 16, i = l % 16) holds K[key i][16 c + 4 g ..
//     + 3] and q[row i] alike; value r of the result is key 4 g + r of row i.
//     O^T += V^T P^T: step r contracts key 4 g + r, whose P is this lane's
//     value r; the lane holds V[key 4 g + r][4 (i + 16 h) .. + 3], component e
//     feeding O block 4 h + e, so O value r' of that block is d = 4 (4 g + r'
//     + 16 h) + e.
//   * Each wavefront keeps its own lazily moved reference max (as
//     sdpa_fwd_kernel), sum and O; the four meet in LDS, and the workgroups'
//     results in sdpa_combine.  Fixed split and order: deterministic.
// Measured, same box (us): 8 x 32 heads on 8 key/value heads, 1 query, 4096
// keys, D 128, against sdpa_fwd_kernel: 703 -> 57 (4.7 TB/s of K and V); error against 64 bits
// 1.2e-6 -> 4.6e-7 (the splits shorten the f32 sums).
#include "bch_internal.h"

#include <math.h>

#include <algorithm>
#include <type_traits>

namespace {

using bch::f32x4;

constexpr float kLog2E = 1.44269504088896340736f;
constexpr float kLazy = 8.0f;      // log2 headroom before the reference max moves
constexpr int kRows = 16;          // query rows per workgroup
constexpr int kBlk = 16;           // keys per block
constexpr int kWaves = 4;

__device__ __forceinline__ float quad_max(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float quad_sum(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// DP: 64 or 128, the head dimension rounded up; FULL: D == DP.
template <int DP, bool FULL>
__global__ __launch_bounds__(64 * kWaves, 2) void sdpa_decode_kernel(
    int H, int Hkv, int Sq, int Skv, int D, float qscale, int rblocks, int splits, int keys_per_split,
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v, float* __restrict__ o,
    bch::SdpaStrides st, float* __restrict__ part) {
  constexpr int NC = DP / 16, NH = DP / 64;
  __shared__ float red_m[kWaves][kRows], red_l[kWaves][kRows];
  __shared__ float red_o[kWaves - 1][kRows][DP + 4];

  // row blocks of one split are neighbours on one XCD (round-robin dispatch over 8), sharing
  // its L2's copy of the keys
  const int nb = gridDim.x;
  int L = blockIdx.x;
  if ((nb & 7) == 0) L = (L & 7) * (nb >> 3) + (L >> 3);
  const int rb = L % rblocks;
  const int sp = L / rblocks % splits;
  const int bk = L / rblocks / splits;
  const int bi = bk / Hkv, hk = bk - bi * Hkv;
  const int group = H / Hkv, rows = group * Sq;

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, g = lane >> 4;
  const float* kh = k + bi * st.k.batch + hk * st.k.head;
  const float* vh = v + bi * st.v.batch + hk * st.v.head;

  // ---- q of row rb * 16 + i (rows past the end repeat the last one and are not stored) ----
  const int row = min(rb * kRows + i, rows - 1);
  const float* qr = q + bi * st.q.batch + (long long)(hk * group + row / Sq) * st.q.head + (row % Sq) * st.q.row;
  f32x4 qf[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int d0 = 16 * c + 4 * g;
    const bool in = FULL || d0 < D;
    const f32x4 x = *reinterpret_cast<const f32x4*>(qr + (in ? d0 : 0));
#pragma unroll
    for (int e = 0; e < 4; ++e) qf[c][e] = in ? x[e] * qscale : 0.0f;
  }

  f32x4 acc[4 * NH];
#pragma unroll
  for (int b = 0; b < 4 * NH; ++b) acc[b] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m_ref = -INFINITY, l_run = 0.0f;

  const int k_begin = sp * keys_per_split, k_end = min(Skv, k_begin + keys_per_split);

  f32x4 kf[2][NC], vf[2][4 * NH];
  // Rows past the last key read it again; FULL unset also past D (zeroed where they are used).
  auto load = [&](int s, int kb) {
    const int key = min(kb + i, Skv - 1);
    const float* kr = kh + (long long)key * st.k.row;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int d0 = 16 * c + 4 * g;
      kf[s][c] = *reinterpret_cast<const f32x4*>(kr + (FULL || d0 < D ? d0 : 0));
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float* vr = vh + (long long)min(kb + 4 * g + r, Skv - 1) * st.v.row;
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        const int d0 = 4 * (i + 16 * h);
        vf[s][r * NH + h] = *reinterpret_cast<const f32x4*>(vr + (FULL || d0 < D ? d0 : 0));
      }
    }
  };
  auto block = [&](int s, int kb) {
    const bool tail = kb + kBlk > Skv;  // uniform
    f32x4 sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      f32x4 kx = kf[s][c];
      if (!FULL) {
        const bool in = 16 * c + 4 * g < D;
#pragma unroll
        for (int e = 0; e < 4; ++e) kx[e] = in ? kx[e] : 0.0f;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) sc = __builtin_amdgcn_mfma_f32_16x16x4f32(kx[e], qf[c][e], sc, 0, 0, 0);
    }
    if (tail) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (kb + 4 * g + r >= Skv) {
          sc[r] = -INFINITY;
#pragma unroll
          for (int h = 0; h < NH; ++h) vf[s][r * NH + h] = (f32x4){0.f, 0.f, 0.f, 0.f};
        }
      }
    }
    const float bm = quad_max(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])));
    const bool move = bm > m_ref + kLazy;  // -inf reference: any finite block max moves it
    if (__any(move)) {
      const float m_new = move ? bm : m_ref;
      const float alpha = m_ref == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_ref - m_new);
      l_run *= alpha;
#pragma unroll
      for (int b = 0; b < 4 * NH; ++b) acc[b] *= alpha;
      m_ref = m_new;
    }
    const float m_use = m_ref == -INFINITY ? 0.0f : m_ref;
    float rs = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      sc[r] = __builtin_amdgcn_exp2f(sc[r] - m_use);
      rs += sc[r];
    }
    l_run += quad_sum(rs);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[4 * h + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[s][r * NH + h][e], sc[r], acc[4 * h + e], 0, 0, 0);
  };

  // wavefront w takes blocks w, w + 4, ... of the split; loads of the block after the last one
  // repeat it
  const int last = k_begin + (k_end - k_begin - 1) / kBlk * kBlk;
  int kb = k_begin + wave * kBlk;
  if (kb < k_end) {
    load(0, kb);
    for (; kb < k_end; kb += 2 * kWaves * kBlk) {
      load(1, min(kb + kWaves * kBlk, last));
      block(0, kb);
      if (kb + kWaves * kBlk >= k_end) break;
      load(0, min(kb + 2 * kWaves * kBlk, last));
      block(1, kb + kWaves * kBlk);
    }
  }

  // ---- the four wavefronts' results, in wavefront order ----
  if (g == 0) {
    red_m[wave][i] = m_ref;
    red_l[wave][i] = l_run;
  }
  if (wave > 0) {
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int r = 0; r < 4; ++r) red_o[wave - 1][i][4 * (4 * g + r + 16 * h) + e] = acc[4 * h + e][r];
  }
  __syncthreads();
  if (wave > 0) return;
  float m = red_m[0][i];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) m = fmaxf(m, red_m[w][i]);
  const float m_use = m == -INFINITY ? 0.0f : m;
  float l = 0.0f;
  float a[kWaves];
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    a[w] = __builtin_amdgcn_exp2f(red_m[w][i] - m_use);
    l += a[w] * red_l[w][i];
  }
#pragma unroll
  for (int b = 0; b < 4 * NH; ++b) acc[b] *= a[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w)
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[4 * h + e][r] += a[w] * red_o[w - 1][i][4 * (4 * g + r + 16 * h) + e];

  const int my = rb * kRows + i;
  if (my >= rows) return;
  float* dst;
  float inv = 1.0f;
  if (splits > 1) {
    float* p = part + ((long long)bk * splits + sp) * bch::sdpa_part_floats(rows, D);
    dst = p + (long long)my * D;
    if (g == 0) {
      p[(long long)rows * D + 2 * my] = m;
      p[(long long)rows * D + 2 * my + 1] = l;
    }
  } else {
    dst = o + bi * st.o.batch + (long long)(hk * group + my / Sq) * st.o.head + (my % Sq) * st.o.row;
    inv = 1.0f / l;
  }
#pragma unroll
  for (int h = 0; h < NH; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d0 = 4 * (4 * g + r + 16 * h);
      if (FULL || d0 < D) {
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[d0 + e] = acc[4 * h + e][r] * inv;
      }
    }
}

// o[row] = sum over splits of 2^(m_s - m) O_s / sum of 2^(m_s - m) l_s, in split order: a
// wavefront per row, lane d (and d + 64).  Two trips to memory bound it: lane s reads split s's
// maximum and sum (at most 64 splits), and the rows of eight splits are loaded before they are
// added, then of four, two and one (8 splits of 256 rows, the two launches: each split's three loads
// in turn 57.8 us, its row in turn 57.1, this 53.5).  Lanes past D read its last column: with a guard
// a load, 14832 rows of D = 32 in few splits took 5.5 us more (the call 24.9 -> 30.3 us, here 25.2).
__global__ __launch_bounds__(64) void sdpa_combine(int H, int Hkv, int Sq, int D, int splits,
                                                   const float* __restrict__ part, float* __restrict__ o,
                                                   bch::SdpaLayout lo) {
  const int group = H / Hkv, rows = group * Sq;
  const int bk = blockIdx.x / rows, row = blockIdx.x % rows;
  const int bi = bk / Hkv, hk = bk - bi * Hkv;
  const long long per = bch::sdpa_part_floats(rows, D);
  const float* p = part + (long long)bk * splits * per;
  const float* ml = p + (long long)rows * D + 2 * row;
  const int lane = threadIdx.x;
  const float ms = lane < splits ? ml[lane * per] : -INFINITY, ls = lane < splits ? ml[lane * per + 1] : 0.0f;
  const float m = bch::wave_allreduce(ms, bch::OpMax());
  const float as = __builtin_amdgcn_exp2f(ms - (m == -INFINITY ? 0.0f : m));
  const int d0 = lane, d1 = lane + 64;
  const float* po = p + (long long)row * D;
  const float *p0 = po + min(d0, D - 1), *p1 = po + min(d1, D - 1);
  const bool wide = D > 64;
  float l = 0.0f, x = 0.0f, y = 0.0f;
  int s = 0;
  // the next U splits, their rows loaded before they are added
  auto add = [&](auto width) {
    constexpr int U = decltype(width)::value;
    float vx[U], vy[U];
#pragma unroll
    for (int u = 0; u < U; ++u) vx[u] = p0[(s + u) * per];
    if (wide) {
#pragma unroll
      for (int u = 0; u < U; ++u) vy[u] = p1[(s + u) * per];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float a = bch::readlane(as, s + u);
      l += a * bch::readlane(ls, s + u);
      x += a * vx[u];
      if (wide) y += a * vy[u];
    }
    s += U;
  };
  while (s + 8 <= splits) add(std::integral_constant<int, 8>{});
  if (s + 4 <= splits) add(std::integral_constant<int, 4>{});
  if (s + 2 <= splits) add(std::integral_constant<int, 2>{});
  if (s < splits) add(std::integral_constant<int, 1>{});
  const float inv = 1.0f / l;
  float* dst = o + bi * lo.batch + (long long)(hk * group + row / Sq) * lo.head + (row % Sq) * lo.row;
  if (d0 < D) dst[d0] = x * inv;
  if (d1 < D) dst[d1] = y * inv;
}

// Two workgroups per CU fill the chip's loads; a split keeps at least 128 keys (two blocks a
// wavefront) and there are at most 64, whose results one wavefront still adds quickly.
struct DecodePlan {
  int rblocks, splits, keys;
};
DecodePlan plan(int B, int H, int Hkv, int Sq, int Skv, bool may_split) {
  DecodePlan p;
  p.rblocks = ((H / Hkv) * Sq + kRows - 1) / kRows;
  const long long units = (long long)B * Hkv * p.rblocks;
  long long want = may_split ? (2LL * bch::device_cu_count() + units - 1) / units : 1;
  want = std::max(1LL, std::min({want, (long long)(Skv / 128), 64LL}));
  p.keys = (int)(((Skv + want - 1) / want + 63) / 64 * 64);
  p.splits = (Skv + p.keys - 1) / p.keys;
  return p;
}

bool mult4(const bch::SdpaLayout& l) { return l.batch % 4 == 0 && l.head % 4 == 0 && l.row % 4 == 0; }
bool aligned16(const float* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

namespace bch {

bool sdpa_decode_applies(int B, int H, int Hkv, int Sq, int Skv, int D, int causal, const float* q, const float* k,
                         const float* v, const SdpaStrides& st) {
  if (causal || D > 128 || D % 4 != 0 || Skv < 128 || (long long)(H / Hkv) * Sq > 128) return false;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !mult4(st.q) || !mult4(st.k) || !mult4(st.v)) return false;
  const DecodePlan p = plan(B, H, Hkv, Sq, Skv, true);
  return Sq <= 16 && (long long)B * Hkv * p.rblocks * p.splits <= 0x7fffffffLL &&
         (long long)B * H * Sq <= 0x7fffffffLL;
}

size_t sdpa_decode_workspace_bytes(int B, int H, int Hkv, int Sq, int Skv, int D) {
  const DecodePlan p = plan(B, H, Hkv, Sq, Skv, true);
  return p.splits > 1 ? sizeof(float) * (size_t)B * Hkv * p.splits * bch::sdpa_part_floats((H / Hkv) * Sq, D) : 0;
}

hipError_t launch_sdpa_decode(hipStream_t s, int B, int H, int Hkv, int Sq, int Skv, int D, float scale,
                              const float* q, const float* k, const float* v, float* o, const SdpaStrides& st,
                              void* ws, size_t ws_bytes) {
  const bool split = ws_bytes >= sdpa_decode_workspace_bytes(B, H, Hkv, Sq, Skv, D);
  const DecodePlan p = plan(B, H, Hkv, Sq, Skv, split);
  const unsigned grid = (unsigned)((long long)B * Hkv * p.rblocks * p.splits);
  float* part = static_cast<float*>(ws);
#define BCH_DECODE(DP_, FULL_)                                                                                    \
  hipLaunchKernelGGL((sdpa_decode_kernel<DP_, FULL_>), dim3(grid), dim3(64 * kWaves), 0, s, H, Hkv, Sq, Skv, D,   \
                     scale * kLog2E, p.rblocks, p.splits, p.keys, q, k, v, o, st, part)
  if (D == 128) BCH_DECODE(128, true);
  else if (D > 64) BCH_DECODE(128, false);
  else if (D == 64) BCH_DECODE(64, true);
  else BCH_DECODE(64, false);
#undef BCH_DECODE
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || p.splits == 1) return e;
  return launch_sdpa_combine(s, B, H, Hkv, Sq, D, p.splits, part, o, st.o);
}

hipError_t launch_sdpa_combine(hipStream_t s, int B, int H, int Hkv, int Sq, int D, int splits, const float* part,
                               float* o, const SdpaLayout& lo) {
  hipLaunchKernelGGL(sdpa_combine, dim3((unsigned)((long long)B * H * Sq)), dim3(64), 0, s, H, Hkv, Sq, D, splits, part,
                     o, lo);
  return hipGetLastError();
}

}  // namespace bch

// sgemm_reserve.hip -- the workspace that a GEMM call has to find where none may be allocated (host).
//
// A call made under capture may not grow the context's workspace (bch_ctx_stream): it is refused
// where it would have to.  Programs size the workspace once, by an eager call or bch_ctx_reserve,
// and capture later, so which calls are refused, and with how much workspace, must not move each
// time a kernel gets faster and the plans of sgemm_mfma.hip with it.  This rule is therefore fixed,
// apart from those plans: the workspace of split-K in equal slices of whole 32-k tiles, of the
// hybrid and of the mixed plan as a v_mfma_f32_32x32x2_f32 kernel would choose them (7.4 us per
// 256 x 256 tile of 32 k), and of the skinny kernels.  A call that finds that much runs, whatever
// its plan would like: every plan but the skinny kernels' takes fewer slices, or none, within the
// workspace at hand.
#include "bch_internal.h"

#include <algorithm>

namespace {

constexpr int kBK = 32, kMinKt = 8;
constexpr double kKtUs = 7.4;
constexpr size_t kMax = (size_t)256 << 20;

struct Opt {
  int bm, bn;
  double eff;
};
constexpr Opt kOpts[] = {{256, 256, 1.0}, {256, 128, 0.966}, {128, 128, 0.92}};

long long tiles_of(const Opt& o, int batch, int m, int n) {
  return (long long)batch * ((m + o.bm - 1) / o.bm) * ((n + o.bn - 1) / o.bn);
}
long long rounds_of(long long wgs) {
  const long long cu = bch::device_cu_count();
  return (wgs + cu - 1) / cu;
}

const Opt& pick(int batch, int m, int n) {
  const Opt* best = nullptr;
  double cost = 0.0;
  for (const Opt& o : kOpts) {
    const double c = (double)rounds_of(tiles_of(o, batch, m, n)) * o.bm * o.bn / o.eff;
    if (best == nullptr || c < cost * 0.999) {
      best = &o;
      cost = c;
    }
  }
  return *best;
}

// Slices of split-K, 1 for none; us: the time modelled.
int slices(int batch, int m, int n, int k, size_t cap, double* us = nullptr) {
  if (batch < 1 || k <= 0 || k % kBK != 0) return 1;
  const Opt& o = pick(batch, m, n);
  const long long tiles = tiles_of(o, batch, m, n);
  if (tiles >= bch::device_cu_count()) return 1;
  const double tk = kKtUs * o.bm * o.bn / 65536.0 / o.eff, mn = (double)batch * m * n * sizeof(float);
  const int nk = k / kBK;
  double best = nk * tk;
  int s = 1;
  for (int sl = 2; nk / sl >= kMinKt; ++sl) {
    if (nk % sl != 0) continue;
    if ((size_t)sl * batch * m * n * sizeof(float) > cap) break;
    const double c = (double)rounds_of(tiles * sl) * (nk / sl) * tk + (2.0 * sl + 1.0) * mn / 5e6 + 2.0;
    if (c < best) {
      best = c;
      s = sl;
    }
  }
  if (us) *us = best;
  return s;
}

// Bytes of the hybrid plan, 0 where it is not taken; us as above.
size_t hybrid(int m, int n, int k, double* us = nullptr) {
  const long long cu = bch::device_cu_count();
  const int nk = k / kBK;
  double dp = 0.0, best = 0.0;
  size_t bytes = 0;
  for (const Opt& o : kOpts) {
    const long long t = tiles_of(o, 1, m, n), rounds = t / cu, r = t % cu;
    const double per = o.bm * o.bn / 65536.0 / o.eff;
    const double c = (double)rounds_of(t) * nk * per;
    if (dp == 0.0 || c < dp) dp = c;
    if (rounds < 1 || r == 0) continue;
    for (int sl = 8; sl >= 2; --sl) {
      const size_t b = (size_t)sl * r * o.bm * o.bn * sizeof(float);
      if (sl * r > cu || nk % sl != 0 || nk / sl < kMinKt || b > kMax) continue;
      const double h =
          (double)(rounds * nk + nk / sl) * per + (2.0 * sl + 1.0) * r * (o.bm * o.bn / 65536.0) * 0.00709 + 0.3;
      if (bytes == 0 || h < best) {
        best = h;
        bytes = b;
      }
      break;
    }
  }
  const bool use = bytes != 0 && best < 0.97 * dp;
  if (us) *us = kKtUs * (use ? best : dp);
  return use ? bytes : 0;
}

double tile_us(int m, int n, int k) {  // k % kBK == 0
  double us = 0.0;
  if (slices(1, m, n, k, kMax, &us) > 1) return us;
  hybrid(m, n, k, &us);
  return us;
}

// Tile path; fixed: within the fixed scratch of bch_sgemm_noalloc, without the hybrid plan.
size_t tile_bytes(int batch, int m, int n, int k, bool fixed) {
  if (k <= 0 || k % kBK != 0) return 0;
  const long long cu = bch::device_cu_count();
  const int mt = (m + 255) / 256, nt = (n + 255) / 256, nk = k / kBK;
  int rm = m, rn = n;  // the mixed plan's rest
  if (batch == 1 && (long long)mt * nt >= cu) {
    double best = 0.99 * tile_us(m, n, k);
    for (int axis = 0; axis < 2; ++axis) {
      const int along = axis == 0 ? mt : nt, across = axis == 0 ? nt : mt;
      for (long long j = (long long)mt * nt / cu; j >= 1; --j) {
        const long long c = j * cu / across;
        if (c < 1 || c >= along) continue;
        const int split = (int)(256 * c), m2 = axis == 0 ? m - split : m, n2 = axis == 0 ? n : n - split;
        const double us = (double)rounds_of(c * across) * nk * kKtUs + tile_us(m2, n2, k) + 16.0;
        if (us < best) {
          best = us;
          rm = m2;
          rn = n2;
        }
      }
    }
  }
  const int sl = slices(batch, rm, rn, k, fixed ? bch::kSgemmFixedScratch : kMax);
  if (sl > 1) return (size_t)sl * batch * rm * rn * sizeof(float);
  return fixed || batch != 1 ? 0 : hybrid(rm, rn, k);
}

}  // namespace

namespace bch {

size_t sgemm_reserved_bytes(bool transb, int batch, int m, int n, int k, int lda, int ldb, bool fixed) {
  if (batch == 1 && !transb && sgemm_skinny_applies(m, n, k, nullptr, k, nullptr, n)) {
    const size_t b = sgemm_skinny_workspace_bytes(m, n, k);
    // 32 < m <= 64 takes the tile path where the skinny partials exceed the fixed scratch
    if (!fixed || m <= 32 || b <= kSgemmFixedScratch) return b;
  }
  if (batch == 1 && transb) {
    if (sgemm_skinny_nt_applies(m, n, k, nullptr, lda, nullptr, ldb)) return sgemm_skinny_nt_workspace_bytes(m, n, k);
    // 33 to 64 rows as two passes of the 32-row kernels
    if (m > 32 && m <= 64 && n >= 8192 && sgemm_skinny_nt_applies(32, n, k, nullptr, lda, nullptr, ldb))
      return std::max(sgemm_skinny_nt_workspace_bytes(32, n, k), sgemm_skinny_nt_workspace_bytes(m - 32, n, k));
  }
  return tile_bytes(batch, m, n, k, fixed);
}

}  // namespace bch

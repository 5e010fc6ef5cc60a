// Device helpers shared by the per-walker kernels: complex arithmetic, wave
// reductions, the register Gauss-Jordan panel and the phaseless weight.
#pragma once
#include <hip/hip_runtime.h>

namespace afq {
namespace wm {

__device__ inline double2 cmul(double2 a, double2 b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
__device__ inline double2 cadd(double2 a, double2 b) { return {a.x + b.x, a.y + b.y}; }
__device__ inline double2 cdiv(double2 a, double2 b) {
  // Smith's algorithm
  if (fabs(b.x) >= fabs(b.y)) {
    const double r = b.y / b.x, den = b.x + b.y * r;
    return {(a.x + a.y * r) / den, (a.y - a.x * r) / den};
  }
  const double r = b.x / b.y, den = b.x * r + b.y;
  return {(a.x * r + a.y) / den, (a.y * r - a.x) / den};
}
__device__ inline double2 cexp(double2 z) {
  const double e = exp(z.x);
  double s, c;
  sincos(z.y, &s, &c);
  return {e * c, e * s};
}

// 1 / (a.x + i a.y) without branches or divisions: conj(a) / |a|^2 on a
// scaled by the power of two 2^-e (exact) that brings max(|re|, |im|) into
// [0.5, 1), so |a|^2 can neither overflow nor underflow; 1 / |a|^2 from the
// hardware reciprocal and two Newton steps (within about an ulp).
__device__ inline double2 crecip_fast(double2 a) {
  const int e = __builtin_amdgcn_frexp_exp(fmax(fabs(a.x), fabs(a.y)));
  const double xs = __builtin_amdgcn_ldexp(a.x, -e), ys = __builtin_amdgcn_ldexp(a.y, -e);
  const double q = fma(xs, xs, ys * ys);
  double r = __builtin_amdgcn_rcp(q);
  r = fma(r, fma(-q, r, 1.0), r);
  r = fma(r, fma(-q, r, 1.0), r);
  const double rs = __builtin_amdgcn_ldexp(r, -e);
  return {xs * rs, -ys * rs};
}

__device__ inline double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

__device__ __forceinline__ double readlane_d(double x, int l) {
  const long long v = __double_as_longlong(x);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(v & 0xffffffffLL), l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(v >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// max(v, v of the lane that DPP control CTRL names), rows outside ROWS kept
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_fmax(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp((int)(b & 0xffffffffLL), (int)(b & 0xffffffffLL), CTRL, ROWS, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), CTRL, ROWS, 0xF, false);
  return fmax(v, __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo)));
}

// maximum of v over the wave (NaN ignored): within quads, half rows and rows,
// then rows 0-1 into row 1 and 2-3 into row 3 (row_bcast 15), rows 0-1 into
// row 3 (row_bcast 31); lane 63 holds the result
__device__ __forceinline__ double wave_fmax(double v) {
  v = dpp_fmax<0xB1, 0xF>(v);   // quad_perm [1, 0, 3, 2]
  v = dpp_fmax<0x4E, 0xF>(v);   // quad_perm [2, 3, 0, 1]
  v = dpp_fmax<0x141, 0xF>(v);  // row_half_mirror
  v = dpp_fmax<0x140, 0xF>(v);  // row_mirror
  v = dpp_fmax<0x142, 0xA>(v);  // row_bcast 15
  v = dpp_fmax<0x143, 0xC>(v);  // row_bcast 31
  return readlane_d(v, 63);
}

// orders a wave's LDS accesses (they are performed in issue order) without a
// work-group barrier
__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Gauss-Jordan steps of one wave on the np <= NP columns a[] of a panel, lane i
// holding the rows i + 64 h of n.  Rows are never swapped: the pivot of column t
// is the first (lowest) not yet used row of maximal |re| + |im| (pj[t], -1 past
// np; `used` marks the rows taken), and column t is replaced by the unit vector
// of its pivot row, so one branch-free update leaves a_p / d in the pivot row
// and a - (f / d) a_p elsewhere.  dp collects the product of the pivots.  The
// pivot row reaches the lanes through scalar registers: it is one of H, and a
// round trip through LDS costs more (H = 2, n = 100: 256 us, 210 without).
template <int H, int NP>
__device__ __forceinline__ void gj_panel(double2 (&a)[H][NP], int np, int n, int lane, unsigned long long (&used)[H],
                                         int (&pj)[NP], double2& dp) {
  static_assert(H == 1 || H == 2, "one or two rows a lane");
#pragma unroll
  for (int t = 0; t < NP; ++t) {
    pj[t] = -1;
    if (t < np) {
      double2 x[H];
      bool cand[H];
      double v[H];
#pragma unroll
      for (int h = 0; h < H; ++h) {
        x[h] = a[h][t];
        cand[h] = lane + 64 * h < n && !((used[h] >> lane) & 1ull);
        v[h] = cand[h] ? fabs(x[h].x) + fabs(x[h].y) : -1.0;
      }
      const double m = wave_fmax(H == 1 ? v[0] : fmax(v[0], v[H - 1]));
      // lowest row of maximal measure (a column of NaNs falls back to the
      // lowest unused row, so p is always a valid row)
      unsigned long long best[H], any = 0;
#pragma unroll
      for (int h = 0; h < H; ++h) {
        best[h] = __ballot(cand[h] && v[h] == m);
        any |= best[h];
      }
#pragma unroll
      for (int h = 0; h < H; ++h)
        if (!any) best[h] = __ballot(cand[h]);
      const bool hi = H > 1 && best[0] == 0;
      const int p = __builtin_ctzll(hi ? best[H - 1] : best[0]);
      pj[t] = hi ? 64 + p : p;
      const double2 xp = {hi ? x[H - 1].x : x[0].x, hi ? x[H - 1].y : x[0].y};
      const double2 d = {readlane_d(xp.x, p), readlane_d(xp.y, p)};
      dp = cmul(dp, d);
      // column t becomes the unit vector of row p: the common update
      // below then leaves 1 / d in row p and -f / d in the others
      const double2 dinv = crecip_fast(d);
      double2 g[H];
      double sc[H];
#pragma unroll
      for (int h = 0; h < H; ++h) {
        const bool isp = lane == p && hi == (h == 1);
        used[h] |= hi == (h == 1) ? 1ull << p : 0ull;
        a[h][t] = isp ? double2{1.0, 0.0} : double2{0.0, 0.0};
        sc[h] = isp ? 0.0 : 1.0;
        const double2 fd = cmul(x[h], dinv);
        g[h] = isp ? dinv : double2{-fd.x, -fd.y};
      }
#pragma unroll
      for (int s = 0; s < NP; ++s) {
        const double2 z = {hi ? a[H - 1][s].x : a[0][s].x, hi ? a[H - 1][s].y : a[0][s].y};
        const double2 r = {readlane_d(z.x, p), readlane_d(z.y, p)};
#pragma unroll
        for (int h = 0; h < H; ++h) {
          const double2 y = a[h][s];
          a[h][s].x = fma(g[h].x, r.x, fma(-g[h].y, r.y, sc[h] * y.x));
          a[h][s].y = fma(g[h].x, r.y, fma(g[h].y, r.x, sc[h] * y.y));
        }
      }
    }
  }
}

// sign of the permutation piv of n <= 128 (in LDS) as true for odd, by one wave:
// the parity of its inversions
__device__ inline bool odd_permutation(const int* piv, int n, int lane) {
  int odd = 0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int i = lane + 64 * h;
    const int pi = i < n ? piv[i] : -1;
#pragma unroll 8
    for (int m = 1; m < n; ++m) odd += m > i && piv[m] < pi;
  }
  return __popcll(__ballot(odd & 1)) & 1;
}

// Phaseless factor |I| cos(theta) (propagation.py:306-320), not clipped, of a
// walker whose overlap went from oo to on, at the population-control shift pcs.
__device__ inline double phaseless_factor(double2 on, double2 oo, double2 sh, double2 ft, double pcs, double2 h0p,
                                          double dt) {
  const double sqdt = sqrt(dt);
  const double2 ratio = cdiv(on, oo);
  const double2 arg = {-sqdt * sh.x + ft.x + dt * (pcs + h0p.x), -sqdt * sh.y + ft.y + dt * h0p.y};
  const double2 imp = cmul(cexp(arg), ratio);
  const double2 ph_arg = cmul(cexp(double2{-sqdt * sh.x, -sqdt * sh.y}), ratio);
  const double theta = atan2(ph_arg.y, ph_arg.x);
  return hypot(imp.x, imp.y) * cos(theta);
}
// The new weight from that factor and the old weight (propagation.py:321-331).
__device__ inline double clipped_weight(double ph, double wt) {
  if (isnan(ph)) ph = 0.0;
  if (ph < 1.0e-3) ph = 0.0;
  if (ph > 100.0) ph = 0.0;
  const double wn = ph * wt;
  return wn > 100.0 ? 0.0 : wn;
}

}  // namespace wm
}  // namespace afq

// Per-walker FP64 dense linear algebra kept in LDS / L2:
//   * Gauss-Jordan determinant + inverse of the O x O overlap matrix T^H W
//     (replaces jnp.linalg.det / jnp.linalg.inv, ad_afqmc/wavefunctions.py:1066,
//     1100, 1266-1268, 1306-1311)
//   * upper Cholesky factor of the O x O Gram matrix W^H W, the middle step of
//     the Cholesky-QR re-orthonormalisation of the block loop (replaces the
//     batched Householder QR of ad_afqmc/linalg_utils.py:51-72; R is
//     discarded there)
//   * CGS2 re-orthonormalisation of an N x O walker panel, kept for the
//     job-free walker entry point, where no Gram or triangle workspace exists.
#include "afq_internal.h"
#include "group.h"
#include "wave_math.h"

namespace afq {
namespace {

using wm::cmul;
using wm::wave_lds_sync;

__device__ inline double2 crecip(double2 a) {
  // Smith's algorithm for 1/(a.x + i a.y)
  if (fabs(a.x) >= fabs(a.y)) {
    const double r = a.y / a.x, den = a.x + a.y * r;
    return {1.0 / den, -r / den};
  }
  const double r = a.x / a.y, den = a.x * r + a.y;
  return {r / den, -1.0 / den};
}

// Gauss-Jordan determinant and inverse, one work-group per matrix,
// partial pivoting on the largest |re|+|im| of the pivot column (LAPACK
// izamax measure).  blockIdx.y selects one of up to two matrix sets (the two
// spins' overlap matrices factor in one launch, so a CU holds two work-groups
// at W = 256).
//
// n <= 128 (gj_reg_body): the matrix stays in registers.  Lane i of every wave
// holds row i, and row i + 64 where n > 64, wave w the columns 8 w .. 8 w + 7
// (one panel).  Rows are never swapped: the pivot of column k is the first
// (lowest) not yet used row of maximal measure (a DPP maximum and a ballot).
// Panel P is factored by wave P alone, column by column, on its own columns
// (the pivot row through scalar registers; column k replaced by the unit vector
// of its pivot row, so one branch-free update leaves a_p / d in the pivot row and
// a - (f / d) a_p elsewhere).  The panel's steps compose to
// M = I + sum_t U_t e_{p_t}^T, and because of the unit vectors the panel's
// columns end up holding M e_{p_t}: after one barrier every other wave applies M
// to its columns as one rank-8 update, a += U a[p_t] (rows p_t as they were
// before the panel).  One barrier a panel instead of one a column.  The result R
// relates to the inverse through the pivot sequence piv (row piv[m] was the
// pivot of column m): A^-1[pinv[r]][piv[c]] = R[r][c], pinv the inverse
// permutation; det A = sign(piv) prod of the pivots (the determinant alone runs
// the same sweep).
//
// Bound by the chain of panel steps and updates (some 0.4 us a column and 2 us a
// panel).  Panels of 8 columns on 8 waves, against 16 on 4: n=20, 256 matrices
// 30 -> 20 us; n=40, 512 57 -> 43; n=60 and 58, 2 x 256 84 -> 73; n=100, 40
// matrices 210 -> 156 (950 in place in global memory, with a barrier and a round
// trip to L2 for each column); n=82, 48 177 -> 127 (800).  The same steps as a
// loop, one column after another through the registers, were 3-15% slower.  Up to
// n = 16 a work-group is the two waves that have columns: with eight, a CU holds a
// quarter of the matrices (overlaps of 2048 walkers, N=130, n=16: 106 us, and 97 in
// panels of 16; 63 so).
//
// n > 128 (gj_det_inv_body, n <= 256): the matrix is factored in global memory,
// in the inverse's buffer or the set's scratch (it stays in L2), with explicit
// row interchanges (the first row of maximal measure at or below k).  Thread t
// owns the columns t % 64 + 64 c for the rows t/64, t/64 + 4, ..., so the
// elimination needs no index division and reads the pivot row and factor
// column as LDS broadcasts.  With an inverse requested the sweep is
// Gauss-Jordan in place (the inverse ends with its columns permuted by the row
// interchanges, undone at the end); for the determinant alone only the
// trailing rows and columns are eliminated (the pivots, hence the determinant,
// are the same).  NMAX = kDetInvMaxN; each thread covers NMAX / 64 columns
// (and pivot-search rows); n <= 64 matrices of such a launch use dynamic LDS.
constexpr int kTwoN = 16;    // largest n of two waves
constexpr int kLdsN = 64;    // largest n of one register row a lane (and of the LDS Cholesky)
constexpr int kReg2N = 128;  // largest n of two register rows a lane
constexpr int kPanel = 8;    // columns of a wave
constexpr size_t reg_lds(int h, int nw, int nmax) {
  const size_t work = sizeof(double2) * (2 * kPanel * 64 * h + nw * kPanel * kPanel);
  return h == 1 ? std::max(work, sizeof(double2) * nmax * (nmax | 1)) : work;
}
constexpr int det_inv_threads(int nmax) {
  return nmax == kTwoN ? 128 : nmax == kLdsN ? 512 : nmax == kReg2N ? 1024 : 256;
}

// H rows a lane, NW waves (n <= 64 H, 8 NW).  lds: reg_lds(H, NW, n) bytes.
template <int H, int NW>
__device__ __forceinline__ void gj_reg_body(const DetInvSet& set, long b, double2* __restrict__ lds) {
  constexpr int ROWS = 64 * H, NT = 64 * NW;
  double2(*ubuf)[kPanel][ROWS] = reinterpret_cast<double2(*)[kPanel][ROWS]>(lds);  // [2]: U[t][row], by panel parity
  // [NW]: per wave, [column][t] of the panel's pivot rows before the panel
  double2(*prow)[kPanel][kPanel] = reinterpret_cast<double2(*)[kPanel][kPanel]>(lds + 2 * kPanel * ROWS);
  __shared__ double2 pdet[NW];  // product of each panel's pivots
  __shared__ int piv[ROWS], pinv[ROWS];
  const int n = set.n;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c0 = kPanel * wave;  // this wave's first column
  const double2* src = set.S + b * set.strideS;
  double2 a[H][kPanel];
  // one row a lane: through LDS, in rows of an odd number of entries, so that
  // global memory is read in runs (lanes a row apart: 9 of 84 us at n = 60)
  const int ld = n | 1;
  if constexpr (H == 1) {
    for (int e = tid; e < n * n; e += NT) {
      const int r = e / n;
      lds[r * ld + e - r * n] = src[e];
    }
    __syncthreads();
    src = lds;
  }
  const int lsrc = H == 1 ? ld : n;
#pragma unroll
  for (int h = 0; h < H; ++h)
#pragma unroll
    for (int t = 0; t < kPanel; ++t) {
      const int r = lane + 64 * h, c = c0 + t;
      a[h][t] = (r < n && c < n) ? src[r * lsrc + c] : double2{0.0, 0.0};
    }
  if constexpr (H == 1) __syncthreads();
  unsigned long long used[H] = {};  // rows already used as pivots (wave-uniform)
  const int npan = (n + kPanel - 1) / kPanel;
  for (int P = 0; P < npan; ++P) {
    const int np = min(kPanel, n - kPanel * P);
    double2(&U)[kPanel][ROWS] = ubuf[P & 1];
    if (wave == P) {
      // ---- the panel, by this wave alone: Gauss-Jordan steps on its columns
      double2 dp = {1.0, 0.0};
      int pj[kPanel];
      wm::gj_panel(a, np, n, lane, used, pj, dp);
      if (lane == 0) {
        pdet[P] = dp;
#pragma unroll
        for (int t = 0; t < kPanel; ++t)
          if (t < np) piv[kPanel * P + t] = pj[t];
      }
      // the panel's transform M = I + sum_t U_t e_{p_t}^T: column t of the
      // panel now holds M e_{p_t}
#pragma unroll
      for (int t = 0; t < kPanel; ++t)
#pragma unroll
        for (int h = 0; h < H; ++h)
          U[t][lane + 64 * h] = (lane + 64 * h == pj[t]) ? double2{a[h][t].x - 1.0, a[h][t].y} : a[h][t];
    }
    __syncthreads();
    if (wave != P && c0 < n) {
      int jj[H];  // the panel's steps whose pivots are this lane's rows
#pragma unroll
      for (int h = 0; h < H; ++h) jj[h] = -1;
#pragma unroll
      for (int t = 0; t < kPanel; ++t) {
        const int p = t < np ? __builtin_amdgcn_readfirstlane(piv[kPanel * P + t]) : -1;
#pragma unroll
        for (int h = 0; h < H; ++h) {
          used[h] |= p >= 0 && (p >> 6) == h ? 1ull << (p & 63) : 0ull;
          jj[h] = (p == lane + 64 * h) ? t : jj[h];
        }
      }
      // ---- apply the panel to this wave's columns: a += U a[p_t] (rows
      // p_t before the panel, through LDS: the lane holding row p_t writes it)
#pragma unroll
      for (int h = 0; h < H; ++h)
        if (jj[h] >= 0) {
#pragma unroll
          for (int s = 0; s < kPanel; ++s) prow[wave][s][jj[h]] = a[h][s];
        }
      wave_lds_sync();
#pragma unroll
      for (int t = 0; t < kPanel; ++t) {
        if (t >= np) break;  // uniform
        double2 u[H];
#pragma unroll
        for (int h = 0; h < H; ++h) u[h] = U[t][lane + 64 * h];
#pragma unroll
        for (int s = 0; s < kPanel; ++s) {
          const double2 r = prow[wave][s][t];
#pragma unroll
          for (int h = 0; h < H; ++h) {
            a[h][s].x = fma(u[h].x, r.x, fma(-u[h].y, r.y, a[h][s].x));
            a[h][s].y = fma(u[h].x, r.y, fma(u[h].y, r.x, a[h][s].y));
          }
        }
      }
      wave_lds_sync();
    }
  }
  __syncthreads();  // piv and pdet complete, U and prow read
  if (wave == NW - 1) {  // it has the fewest columns to store
    const bool neg = wm::odd_permutation(piv, n, lane);
    double2 dprod = {1.0, 0.0};
    for (int q = 0; q < npan; ++q) dprod = cmul(dprod, pdet[q]);
    if (lane == 0) set.det[b] = neg ? double2{-dprod.x, -dprod.y} : dprod;
  }
  if (!set.inv) return;
  if (tid < n) pinv[piv[tid]] = tid;
  __syncthreads();
  double2* dst = set.inv + b * set.strideInv;
  double2* out = H == 1 ? lds : dst;
#pragma unroll
  for (int h = 0; h < H; ++h) {
    const int r = lane + 64 * h;
    if (r < n) {
      const long row = (long)pinv[r] * lsrc;
#pragma unroll
      for (int t = 0; t < kPanel; ++t)
        if (c0 + t < n) out[row + piv[c0 + t]] = a[h][t];
    }
  }
  if constexpr (H == 1) {
    __syncthreads();
    for (int e = tid; e < n * n; e += NT) {
      const int r = e / n;
      dst[e] = lds[r * ld + e - r * n];
    }
  }
}

template <int NMAX>
__device__ __forceinline__ void gj_det_inv_body(const DetInvSet& set, long b, double2* __restrict__ lds) {
  constexpr int kColsPer = NMAX / 64;
  __shared__ double2 prow[NMAX];
  __shared__ double2 fcol[NMAX];
  __shared__ int piv[NMAX];
  __shared__ int pk;
  const int n = set.n;
  double2* __restrict__ det = set.det;
  double2* __restrict__ inv = set.inv;
  const int tid = threadIdx.x;
  const int j = tid & 63, rg = tid >> 6;
  const double2* src = set.S + b * set.strideS;
  const int nn = n * n;
  const bool want_inv = inv != nullptr;
  double2* a = lds;
  if (n > kLdsN) a = want_inv ? inv + b * set.strideInv : set.work + b * set.strideS;
  if (a != src)
    for (int i = tid; i < nn; i += 256) a[i] = src[i];
  __syncthreads();

  double2 dprod = {1.0, 0.0};
  bool neg = false;
  for (int k = 0; k < n; ++k) {
    if (tid < 64) {
      double v = -1.0;
      int idx = tid;
#pragma unroll
      for (int m = 0; m < kColsPer; ++m) {
        const int r = tid + 64 * m;
        if (r >= k && r < n) {
          const double2 x = a[r * n + k];
          const double vr = fabs(x.x) + fabs(x.y);
          if (vr > v) {  // rows ascend: a tie keeps the lower row
            v = vr;
            idx = r;
          }
        }
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        const double ov = __shfl_xor(v, off);
        const int oi = __shfl_xor(idx, off);
        if (ov > v || (ov == v && oi < idx)) {
          v = ov;
          idx = oi;
        }
      }
      if (tid == 0) {
        pk = idx;
        piv[k] = idx;
      }
    }
    __syncthreads();
    const int p = pk;
    const double2 d = a[p * n + k];
    const double2 dinv = crecip(d);
    if (tid == 0) {
      dprod = cmul(dprod, d);
      if (p != k) neg = !neg;
    }
    // read: the pivot row (scaled) and the rows to swap (group 0), the factor
    // column after the swap (group 1)
    const int jlo = want_inv ? 0 : k;
    double2 xp[kColsPer], xk[kColsPer], fc[kColsPer];
#pragma unroll
    for (int c = 0; c < kColsPer; ++c) {
      const int jc = j + 64 * c;
      xp[c] = xk[c] = fc[c] = double2{0.0, 0.0};
      if (rg == 0 && jc >= jlo && jc < n) {
        xp[c] = a[p * n + jc];
        xk[c] = a[k * n + jc];
      } else if (rg == 1 && jc < n) {
        fc[c] = (jc == k) ? d : a[(jc == p ? k : jc) * n + k];
      }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kColsPer; ++c) {
      const int jc = j + 64 * c;
      if (rg == 0 && jc >= jlo && jc < n) {
        const double2 r = (jc == k) ? dinv : cmul(xp[c], dinv);
        prow[jc] = r;
        a[k * n + jc] = r;
        if (p != k) a[p * n + jc] = xk[c];
      } else if (rg == 1 && jc < n) {
        fcol[jc] = fc[c];
      }
    }
    __syncthreads();
    const int i0 = want_inv ? rg : k + 1 + rg;
#pragma unroll
    for (int c = 0; c < kColsPer; ++c) {
      const int jc = j + 64 * c;
      if (jc < n && jc >= jlo) {
        const double2 rk = prow[jc];
#pragma unroll 4
        for (int i = i0; i < n; i += 4) {
          if (i == k) continue;
          const double2 f = fcol[i];
          double2* x = &a[i * n + jc];
          if (jc == k) {
            *x = double2{-(f.x * rk.x - f.y * rk.y), -(f.x * rk.y + f.y * rk.x)};
          } else {
            double2 y = *x;
            y.x -= f.x * rk.x - f.y * rk.y;
            y.y -= f.x * rk.y + f.y * rk.x;
            *x = y;
          }
        }
      }
    }
    __syncthreads();
  }
  if (tid == 0) det[b] = neg ? double2{-dprod.x, -dprod.y} : dprod;
  if (inv) {
    // undo the column permutation: each thread owns whole rows, so no barrier
    // is needed between the sequential swaps.
    for (int i = tid; i < n; i += 256) {
      for (int k = n - 1; k >= 0; --k) {
        const int p = piv[k];
        if (p != k) {
          const double2 t = a[i * n + k];
          a[i * n + k] = a[i * n + p];
          a[i * n + p] = t;
        }
      }
    }
    __syncthreads();
    double2* dst = inv + b * set.strideInv;
    if (dst != a)
      for (int i = tid; i < nn; i += 256) dst[i] = a[i];
  }
}

template <int NMAX>
__global__ __launch_bounds__(det_inv_threads(NMAX)) void gj_det_inv_kernel(DetInvSet s0, DetInvSet s1) {
  extern __shared__ double2 lds_gj[];
  if constexpr (NMAX == kTwoN)
    gj_reg_body<1, 2>(blockIdx.y == 0 ? s0 : s1, blockIdx.x, lds_gj);
  else if constexpr (NMAX == kLdsN)
    gj_reg_body<1, 8>(blockIdx.y == 0 ? s0 : s1, blockIdx.x, lds_gj);
  else if constexpr (NMAX == kReg2N)
    gj_reg_body<2, 16>(blockIdx.y == 0 ? s0 : s1, blockIdx.x, lds_gj);
  else
    gj_det_inv_body<NMAX>(blockIdx.y == 0 ? s0 : s1, blockIdx.x, lds_gj);
}

// Grouped: work-group i factors matrix i - prefix[j] of job j's set.
template <int NMAX>
__global__ __launch_bounds__(det_inv_threads(NMAX)) void gj_det_inv_grouped_kernel(
    const DetInvSet* __restrict__ sets, const int* __restrict__ prefix, int njobs) {
  extern __shared__ double2 lds_gj[];
  const int item = blockIdx.x;
  const int j = group_find(prefix, njobs, item);
  const DetInvSet set = sets[j];
  if constexpr (NMAX == kTwoN)
    gj_reg_body<1, 2>(set, item - prefix[j], lds_gj);
  else if constexpr (NMAX == kLdsN)
    gj_reg_body<1, 8>(set, item - prefix[j], lds_gj);
  else if constexpr (NMAX == kReg2N)
    gj_reg_body<2, 16>(set, item - prefix[j], lds_gj);
  else
    gj_det_inv_body<NMAX>(set, item - prefix[j], lds_gj);
}

using wm::wave_sum;

__global__ __launch_bounds__(256) void cgs2_kernel(double2* __restrict__ Wp, long ld, long sW, int nr, int nc) {
  __shared__ double2 r[128];
  __shared__ double red[4];
  double2* Wb = Wp + (long)blockIdx.x * sW;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int j = 0; j < nc; ++j) {
    for (int pass = 0; pass < 2 && j > 0; ++pass) {
      for (int k = wave; k < j; k += 4) {
        double sr = 0.0, si = 0.0;
        for (int p = lane; p < nr; p += 64) {
          const double2 q = Wb[(long)p * ld + k], x = Wb[(long)p * ld + j];
          sr += q.x * x.x + q.y * x.y;
          si += q.x * x.y - q.y * x.x;
        }
        sr = wave_sum(sr);
        si = wave_sum(si);
        if (lane == 0) r[k] = double2{sr, si};
      }
      __syncthreads();
      for (int p = tid; p < nr; p += 256) {
        double2 x = Wb[(long)p * ld + j];
        for (int k = 0; k < j; ++k) {
          const double2 q = Wb[(long)p * ld + k], rk = r[k];
          x.x -= q.x * rk.x - q.y * rk.y;
          x.y -= q.x * rk.y + q.y * rk.x;
        }
        Wb[(long)p * ld + j] = x;
      }
      __syncthreads();
    }
    double s = 0.0;
    for (int p = tid; p < nr; p += 256) {
      const double2 x = Wb[(long)p * ld + j];
      s += x.x * x.x + x.y * x.y;
    }
    s = wave_sum(s);
    if (lane == 0) red[wave] = s;
    __syncthreads();
    const double scale = 1.0 / sqrt(red[0] + red[1] + red[2] + red[3]);
    for (int p = tid; p < nr; p += 256) {
      double2 x = Wb[(long)p * ld + j];
      x.x *= scale;
      x.y *= scale;
      Wb[(long)p * ld + j] = x;
    }
    __syncthreads();
  }
}

// Upper Cholesky factor R (S = R^H R, positive real diagonal) of `count`
// Hermitian positive-definite n x n matrices (n <= 256), one 256-thread
// work-group per matrix, in dynamic LDS up to n = 64 and in place in R above;
// thread t owns the columns t % 64 + 64 c for the rows t/64, t/64 + 4, ...
// The strict lower triangle of R is written as zero.
template <int NMAX>
__device__ __forceinline__ void cholesky_upper_body(const double2* __restrict__ S, long strideS, int n,
                                                    double2* __restrict__ R, long strideR, long b,
                                                    double2* __restrict__ lds) {
  constexpr int kColsPer = NMAX / 64;
  const int tid = threadIdx.x;
  const int j = tid & 63, rg = tid >> 6;
  const double2* src = S + b * strideS;
  double2* dst = R + b * strideR;
  const int nn = n * n;
  double2* a = lds;
  if constexpr (NMAX > kLdsN)
    if (n > kLdsN) a = dst;
  if (a != src)
    for (int i = tid; i < nn; i += 256) a[i] = src[i];
  __syncthreads();
  for (int k = 0; k < n; ++k) {
    const double dinv = 1.0 / sqrt(a[k * n + k].x);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kColsPer; ++c) {
      const int jc = j + 64 * c;
      if (rg == 0 && jc >= k && jc < n) {
        const double2 x = a[k * n + jc];
        a[k * n + jc] = (jc == k) ? double2{1.0 / dinv, 0.0} : double2{x.x * dinv, x.y * dinv};
      }
    }
    __syncthreads();
    if constexpr (NMAX == kLdsN) {
      // reads first, then the updates (as in the Gauss-Jordan sweep)
      if (j > k && j < n) {
        const double2 rkj = a[k * n + j];
        double2 xv[16], rv[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) {
          const int i = k + 1 + rg + 4 * t;
          xv[t] = rv[t] = double2{0.0, 0.0};
          if (i <= j) {
            rv[t] = a[k * n + i];
            xv[t] = a[i * n + j];
          }
        }
#pragma unroll
        for (int t = 0; t < 16; ++t) {
          const int i = k + 1 + rg + 4 * t;
          if (i <= j) {  // S_ij -= conj(R_ki) R_kj
            xv[t].x -= rv[t].x * rkj.x + rv[t].y * rkj.y;
            xv[t].y -= rv[t].x * rkj.y - rv[t].y * rkj.x;
            a[i * n + j] = xv[t];
          }
        }
      }
    } else {
#pragma unroll
      for (int c = 0; c < kColsPer; ++c) {
        const int jc = j + 64 * c;
        if (jc > k && jc < n) {
          const double2 rkj = a[k * n + jc];
          for (int i = k + 1 + rg; i <= jc; i += 4) {
            const double2 rki = a[k * n + i];  // S_ij -= conj(R_ki) R_kj
            double2 x = a[i * n + jc];
            x.x -= rki.x * rkj.x + rki.y * rkj.y;
            x.y -= rki.x * rkj.y - rki.y * rkj.x;
            a[i * n + jc] = x;
          }
        }
      }
    }
    __syncthreads();
  }
  for (int i = tid; i < nn; i += 256) {
    const int r = i / n, c = i - r * n;
    if (c < r)
      dst[i] = double2{0.0, 0.0};
    else if (dst != a)
      dst[i] = a[i];
  }
}

// grid (count, sets): matrix blockIdx.x of set blockIdx.y
template <int NMAX>
__global__ __launch_bounds__(256) void cholesky_upper_kernel(CholSet c0, CholSet c1) {
  extern __shared__ double2 lds_ch[];
  const CholSet c = blockIdx.y == 0 ? c0 : c1;
  cholesky_upper_body<NMAX>(c.S, c.strideS, c.n, c.R, c.strideR, blockIdx.x, lds_ch);
}

template <int NMAX>
__global__ __launch_bounds__(256) void cholesky_grouped_kernel(const CholSet* __restrict__ sets,
                                                              const int* __restrict__ prefix, int njobs) {
  extern __shared__ double2 lds_ch[];
  const int item = blockIdx.x;
  const int j = group_find(prefix, njobs, item);
  const CholSet c = sets[j];
  cholesky_upper_body<NMAX>(c.S, c.strideS, c.n, c.R, c.strideR, item - prefix[j], lds_ch);
}

// Dynamic LDS of the largest of these kernels' launches (64 x 65 entries), and room
constexpr size_t kLdsMax = 96 * 1024;

// Grouped copies / conjugate copies: work-group i covers elements
// [(i - prefix[j]) * 1024, +1024) of job j's vector.
__global__ __launch_bounds__(256) void vec_grouped_kernel(const VecJob* __restrict__ jobs,
                                                          const int* __restrict__ prefix, int njobs) {
  const int item = blockIdx.x;
  const int j = group_find(prefix, njobs, item);
  const VecJob v = jobs[j];
  const long base = (long)(item - prefix[j]) * 1024;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const long i = base + t * 256 + threadIdx.x;
    if (i < v.n) {
      const double2 x = v.src[i];
      v.dst[i] = v.conj ? double2{x.x, -x.y} : x;
    }
  }
}

}  // namespace

// Dynamic LDS of the det/inverse and Cholesky kernels: the largest matrix
// factored in LDS (n <= 64; larger ones are factored in global memory).
static size_t matrix_lds_bytes(int nmax) {
  const int m = std::min(nmax, kLdsN);
  return sizeof(double2) * m * m;
}

static int check_det_inv_set(const DetInvSet& s) {
  if (s.n < 1 || s.n > kDetInvMaxN)
    return fail(AFQ_E_UNSUPPORTED, "det/inverse kernel supports 1 <= n <= " + std::to_string(kDetInvMaxN));
  if (s.n > kLdsN && !s.inv && !s.work)
    return fail(AFQ_E_INVALID, "det/inverse: n > 64 without an inverse needs a scratch matrix per entry");
  return AFQ_OK;
}

template <int NMAX>
static int launch_det_inv(const DetInvSet* sets, int nsets, int count, size_t lds, hipStream_t stream) {
  static std::atomic<uint64_t> raised{0};
  AFQ_TRY(raise_lds(reinterpret_cast<const void*>(gj_det_inv_kernel<NMAX>), kLdsMax, raised, "det/inverse"));
  hipLaunchKernelGGL(gj_det_inv_kernel<NMAX>, dim3(count, nsets), dim3(det_inv_threads(NMAX)), lds, stream, sets[0],
                     sets[nsets > 1 ? 1 : 0]);
  return launch_status("gj_det_inv_kernel");
}

int batched_det_inv_sets(const DetInvSet* sets, int nsets, int count, hipStream_t stream) {
  if (nsets < 1 || nsets > 2) return fail(AFQ_E_INVALID, "det/inverse: one or two matrix sets");
  int nmax = 0;
  for (int i = 0; i < nsets; ++i) {
    AFQ_TRY(check_det_inv_set(sets[i]));
    nmax = std::max(nmax, sets[i].n);
  }
  if (count <= 0) return AFQ_OK;
  // n <= 128: the matrices stay in registers
  return nmax <= kTwoN    ? launch_det_inv<kTwoN>(sets, nsets, count, reg_lds(1, 2, nmax), stream)
         : nmax <= kLdsN  ? launch_det_inv<kLdsN>(sets, nsets, count, reg_lds(1, 8, nmax), stream)
         : nmax <= kReg2N ? launch_det_inv<kReg2N>(sets, nsets, count, reg_lds(2, 16, nmax), stream)
                          : launch_det_inv<kDetInvMaxN>(sets, nsets, count, matrix_lds_bytes(nmax), stream);
}

template <int NMAX>
static int launch_det_inv_grouped(const GroupTab<DetInvSet>& t, size_t lds, hipStream_t stream) {
  static std::atomic<uint64_t> raised{0};
  AFQ_TRY(raise_lds(reinterpret_cast<const void*>(gj_det_inv_grouped_kernel<NMAX>), kLdsMax, raised, "det/inverse"));
  hipLaunchKernelGGL(gj_det_inv_grouped_kernel<NMAX>, dim3((unsigned)t.total), dim3(det_inv_threads(NMAX)), lds, stream, t.params,
                     t.prefix, t.njobs);
  return launch_status("gj_det_inv_grouped_kernel");
}

int det_inv_grouped(const GroupTab<DetInvSet>& t, int nmax, hipStream_t stream) {
  if (t.njobs < 1 || t.total < 1) return AFQ_OK;
  if (nmax < 1 || nmax > kDetInvMaxN)
    return fail(AFQ_E_UNSUPPORTED, "det/inverse kernel supports 1 <= n <= " + std::to_string(kDetInvMaxN));
  return nmax <= kTwoN    ? launch_det_inv_grouped<kTwoN>(t, reg_lds(1, 2, nmax), stream)
         : nmax <= kLdsN  ? launch_det_inv_grouped<kLdsN>(t, reg_lds(1, 8, nmax), stream)
         : nmax <= kReg2N ? launch_det_inv_grouped<kReg2N>(t, reg_lds(2, 16, nmax), stream)
                          : launch_det_inv_grouped<kDetInvMaxN>(t, matrix_lds_bytes(nmax), stream);
}

int batched_det_inv(const double2* S, long strideS, int n, int count, double2* det, double2* inv, long strideInv,
                    hipStream_t stream) {
  const DetInvSet set{S, strideS, n, det, inv, strideInv};
  return batched_det_inv_sets(&set, 1, count, stream);
}

template <int NMAX>
static int launch_cholesky(const CholSet* sets, int nsets, int count, size_t lds, hipStream_t stream) {
  static std::atomic<uint64_t> raised{0};
  AFQ_TRY(raise_lds(reinterpret_cast<const void*>(cholesky_upper_kernel<NMAX>), kLdsMax, raised, "Cholesky"));
  hipLaunchKernelGGL(cholesky_upper_kernel<NMAX>, dim3(count, nsets), dim3(256), lds, stream, sets[0],
                     sets[nsets > 1 ? 1 : 0]);
  return launch_status("cholesky_upper_kernel");
}

int batched_cholesky_upper_sets(const CholSet* sets, int nsets, int count, hipStream_t stream) {
  if (nsets < 1 || nsets > 2) return fail(AFQ_E_INVALID, "Cholesky: one or two matrix sets");
  int nmax = 0;
  for (int i = 0; i < nsets; ++i) {
    if (sets[i].n < 1 || sets[i].n > kDetInvMaxN)
      return fail(AFQ_E_UNSUPPORTED, "Cholesky kernel supports 1 <= n <= " + std::to_string(kDetInvMaxN));
    nmax = std::max(nmax, sets[i].n);
  }
  if (count <= 0) return AFQ_OK;
  const size_t lds = matrix_lds_bytes(nmax);
  return nmax <= kLdsN ? launch_cholesky<kLdsN>(sets, nsets, count, lds, stream)
                       : launch_cholesky<kDetInvMaxN>(sets, nsets, count, lds, stream);
}

int batched_cholesky_upper(const double2* S, long strideS, int n, int count, double2* R, long strideR,
                           hipStream_t stream) {
  const CholSet set{S, strideS, n, R, strideR};
  return batched_cholesky_upper_sets(&set, 1, count, stream);
}

template <int NMAX>
static int launch_cholesky_grouped(const GroupTab<CholSet>& t, size_t lds, hipStream_t stream) {
  static std::atomic<uint64_t> raised{0};
  AFQ_TRY(raise_lds(reinterpret_cast<const void*>(cholesky_grouped_kernel<NMAX>), kLdsMax, raised, "Cholesky"));
  hipLaunchKernelGGL(cholesky_grouped_kernel<NMAX>, dim3((unsigned)t.total), dim3(256), lds, stream, t.params,
                     t.prefix, t.njobs);
  return launch_status("cholesky_grouped_kernel");
}

int cholesky_grouped(const GroupTab<CholSet>& t, int nmax, hipStream_t stream) {
  if (t.njobs < 1 || t.total < 1) return AFQ_OK;
  if (nmax < 1 || nmax > kDetInvMaxN)
    return fail(AFQ_E_UNSUPPORTED, "Cholesky kernel supports 1 <= n <= " + std::to_string(kDetInvMaxN));
  const size_t lds = matrix_lds_bytes(nmax);
  return nmax <= kLdsN ? launch_cholesky_grouped<kLdsN>(t, lds, stream)
                       : launch_cholesky_grouped<kDetInvMaxN>(t, lds, stream);
}

int vec_grouped(const GroupTab<VecJob>& t, hipStream_t stream) {
  if (t.njobs < 1 || t.total < 1) return AFQ_OK;
  hipLaunchKernelGGL(vec_grouped_kernel, dim3((unsigned)t.total), dim3(256), 0, stream, t.params, t.prefix, t.njobs);
  return launch_status("vec_grouped_kernel");
}


int batched_cgs2(double2* Wp, long ld, long sW, int n_rows, int n_cols, int count, hipStream_t stream) {
  if (n_cols < 1 || n_cols > 128 || n_cols > n_rows) return fail(AFQ_E_UNSUPPORTED, "CGS2 supports 1 <= nocc <= 128 <= N");
  if (count <= 0) return AFQ_OK;
  hipLaunchKernelGGL(cgs2_kernel, dim3(count), dim3(256), 0, stream, Wp, ld, sW, n_rows, n_cols);
  return launch_status("cgs2_kernel");
}

}  // namespace afq

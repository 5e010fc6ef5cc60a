// Phaseless step (N <= 48 orbitals) and measurement of small FP64 jobs with at
// most 16 occupied orbitals per spin: one work-group per walker keeps the walker's panel,
// its overlap inverse, Green's function, VHS and Taylor terms in LDS, so a step
// is one launch instead of some seventeen (ad_afqmc/propagation.py:274-336) and
// a measurement's per-walker part another (walkers.py:155-157,
// wavefunctions.py:1064-1100, 1259-1312).
//
// Bound: the latency of each short phase at N ~ 10 (14 us a step of a block at
// N = 10, O = 5, G = 27, 50 walkers, 85 us as separate launches; a block of ten
// steps 1.07 -> 0.32 ms); at the upper end the L2 reads of L and rot_chol, which
// every walker repeats (N = 37, O = 9 / 7, G = 149, 101 walkers: 187 -> 85 us a
// step): small_step_pays draws that line.
#include "small.h"

#include "wave_math.h"

namespace afq {
namespace {

using wm::cadd;
using wm::cmul;
using wm::wave_sum;

// LDS regions in double2: X and Y panels (N x c), V (the VHS; before it the
// Green's functions), E (exp(-dt/2 h1) of every buffer), T, the shifted fields.
struct Regions {
  int ldv, panel, v, e, t;
};
__host__ __device__ inline Regions regions(int N, int c, int osum, int nbuf) {
  Regions r;
  r.ldv = N | 1;  // odd row stride: rows read down a column start in distinct banks
  r.panel = N * c;
  r.v = N * r.ldv;
  if (N * osum > r.v) r.v = N * osum;
  r.e = (nbuf * N * N + 1) / 2;
  r.t = (N * osum + 1) / 2;
  return r;
}
__host__ __device__ inline int vhs_entries(int N, bool sym) { return sym ? N * (N + 1) / 2 : N * N; }

// Row and column of entry e.
__device__ inline void vhs_entry(int e, int N, bool sym, int& i, int& j) {
  if (sym) {
    i = (int)((sqrtf(8.0f * e + 1.0f) - 1.0f) * 0.5f);
    if ((i + 1) * (i + 2) / 2 <= e) ++i;
    if (i * (i + 1) / 2 > e) --i;
    j = e - i * (i + 1) / 2;
  } else {
    i = e / N;
    j = e - i * N;
  }
}

// Sum of v over the work-group, for every thread; red: one element a wave.
template <int NT>
__device__ inline double2 group_sum2(double2 v, double2* red) {
  v.x = wave_sum(v.x);
  v.y = wave_sum(v.y);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double2 r = red[0];
#pragma unroll
  for (int i = 1; i < NT / 64; ++i) r = cadd(r, red[i]);
  return r;
}

template <int NT>
__device__ inline void load_panel(const SmallJob& b, long w, double2* X) {
  int col = 0;
  for (int s = 0; s < b.nbuf; ++s) {
    const int cs = b.cb[s], n = b.N * cs;
    const double2* src = b.wbuf[s] + w * n;
    for (int e = threadIdx.x; e < n; e += NT) X[(e / cs) * b.c + col + e % cs] = src[e];
    col += cs;
  }
}
template <int NT>
__device__ inline void store_panel(const SmallJob& b, long w, const double2* X) {
  int col = 0;
  for (int s = 0; s < b.nbuf; ++s) {
    const int cs = b.cb[s], n = b.N * cs;
    double2* dst = b.wbuf[s] + w * n;
    for (int e = threadIdx.x; e < n; e += NT) dst[e] = X[(e / cs) * b.c + col + e % cs];
    col += cs;
  }
}
// T_s (N x occ_s) of every spin, one after another
template <int NT>
__device__ inline void load_trial(const SmallJob& b, double* T) {
  int at = 0;
  for (int s = 0; s < b.nspin; ++s) {
    const int n = b.N * b.occ[s];
    for (int e = threadIdx.x; e < n; e += NT) T[at + e] = b.mo[s][e];
    at += n;
  }
}

// S_s = T_s^T W_s of every spin
template <int NT>
__device__ inline void overlap_matrices(const SmallJob& b, const double* T, const double2* X, double2 (*S)[256]) {
  const int n0 = b.occ[0] * b.occ[0], n = n0 + (b.nspin > 1 ? b.occ[1] * b.occ[1] : 0);
  for (int e = threadIdx.x; e < n; e += NT) {
    const int s = e >= n0, O = b.occ[s], l = e - s * n0, i = l / O, j = l - i * O;
    const double* t = T + s * b.N * b.occ[0] + i;
    const double2* x = X + b.off[s] + j;
    double2 a = {0.0, 0.0};
#pragma unroll 4
    for (int p = 0; p < b.N; ++p) {
      const double tv = t[p * O];
      const double2 xv = x[p * b.c];
      a.x += tv * xv.x;
      a.y += tv * xv.y;
    }
    S[s][l] = a;
  }
}

// Determinant and inverse (over S) of one wave's n x n matrix, n <= NP.
template <int NP>
__device__ inline void invert_wave(int n, double2* S, double2* det) {
  const int lane = threadIdx.x & 63;
  double2 a[1][NP];
#pragma unroll
  for (int t = 0; t < NP; ++t) a[0][t] = (lane < n && t < n) ? S[lane * n + t] : double2{0.0, 0.0};
  unsigned long long used[1] = {0};
  int pj[NP];
  double2 dp = {1.0, 0.0};
  wm::gj_panel(a, n, n, lane, used, pj, dp);
  int to = 0;  // the column whose pivot is this lane's row
#pragma unroll
  for (int t = 0; t < NP; ++t) to = (t < n && pj[t] == lane) ? t : to;
#pragma unroll
  for (int t = 0; t < NP; ++t)
    if (lane < n && t < n) S[to * n + pj[t]] = a[0][t];
  // parity of the pivot permutation from its inversions, one row a lane
  int odd = 0;
#pragma unroll
  for (int m = 0; m < NP; ++m) odd += m < n && m > to && pj[m] < lane;
  const bool neg = __popcll(__ballot(lane < n && (odd & 1))) & 1;
  if (lane == 0) *det = neg ? double2{-dp.x, -dp.y} : dp;
}

typedef __attribute__((address_space(3))) double2* LdsPtr;

// Out of line: one copy of the unrolled sweeps, which the instruction cache
// holds.
__device__ __attribute__((noinline)) void invert_call(int n, LdsPtr S, LdsPtr det) {
  if (n <= 8)
    invert_wave<8>(n, (double2*)S, (double2*)det);
  else if (n <= 12)
    invert_wave<12>(n, (double2*)S, (double2*)det);
  else
    invert_wave<16>(n, (double2*)S, (double2*)det);
}

// The same for S_s of every spin, wave s for spin s.
__device__ inline void invert(const SmallJob& b, double2 (*S)[256], double2* det) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (wave < b.nspin) invert_call(b.occ[wave], (LdsPtr)S[wave], (LdsPtr)(det + wave));
}

// G_s = (W_s S_s^-1)^T (occ_s x N) of every spin, one after another
template <int NT>
__device__ inline void greens(const SmallJob& b, const double2* X, const double2 (*inv)[256], double2* Gm) {
  const int n0 = b.occ[0] * b.N, n = n0 + (b.nspin > 1 ? b.occ[1] * b.N : 0);
  for (int e = threadIdx.x; e < n; e += NT) {
    const int s = e >= n0, O = b.occ[s], l = e - s * n0, i = l / b.N, p = l - i * b.N;
    const double2* x = X + p * b.c + b.off[s];
    double2 a = {0.0, 0.0};
#pragma unroll 4
    for (int k = 0; k < O; ++k) {
      const double2 u = inv[s][k * O + i], v = x[k];
      a.x += u.x * v.x - u.y * v.y;
      a.y += u.x * v.y + u.y * v.x;
    }
    Gm[e] = a;
  }
}

// The thread's TR x TR tiles of an N x c panel: rows r and r + ceil(N/TR), columns likewise.
template <int NT, int TR, int TPT>
struct Tiles {
  int row[TPT][TR], col[TPT][TR];
  bool on[TPT];
  __device__ Tiles(int N, int c) {
    const int nr = (N + TR - 1) / TR, nc = (c + TR - 1) / TR;
#pragma unroll
    for (int u = 0; u < TPT; ++u) {
      const int t = threadIdx.x + u * NT;
      on[u] = t < nr * nc;
      const int r = on[u] ? t / nc : 0, q = on[u] ? t - r * nc : 0;
#pragma unroll
      for (int i = 0; i < TR; ++i) {
        row[u][i] = r + i * nr;
        col[u][i] = q + i * nc;
      }
    }
  }
};

// Out of line: inlined in the step loop, the constants of exp, sin, cos and
// atan2 would be kept in registers through all of it.
__device__ __attribute__((noinline)) double factor_call(double2 on, double2 oo, double2 sh, double2 ft, double pcs,
                                                        double2 h0p, double dt) {
  return wm::phaseless_factor(on, oo, sh, ft, pcs, h0p, dt);
}

// nsteps steps of walker blockIdx.x.  Nothing in a walker's path depends on the
// weights, so the steps need no exchange between walkers.  With RES, L (the
// entries of one triangle where it is symmetric) and rot_chol sit in LDS for
// all steps; without, every step streams them from L2, about 30 loads a thread
// in flight.
template <int NT, int TR, int TPT, bool RES>
__global__ __launch_bounds__(NT) void small_step_kernel(SmallStep p) {
  extern __shared__ double2 sm[];
  __shared__ double2 S[2][256];
  __shared__ double2 det[2], red[NT / 64];
  const SmallJob& b = p.b;
  const int tid = threadIdx.x;
  const int N = b.N, c = b.c, G = b.G;
  const long w = blockIdx.x, NN = (long)N * N;
  const int occ1 = b.nspin > 1 ? b.occ[1] : 0, osum = b.occ[0] + occ1;
  const Regions rg = regions(N, c, osum, b.nbuf);
  double2* P = sm;
  double2* Q = P + rg.panel;
  double2* V = Q + rg.panel;
  double2* xs = V + rg.v;
  double* E = reinterpret_cast<double*>(xs + G);
  double* T = E + 2 * rg.e;
  const int nent = vhs_entries(N, p.sym), nrc = N * osum;
  const int nl2 = (nent + 1) >> 1, nr2 = (nrc + 1) >> 1;  // pairs a Cholesky index
  double2* Lr = reinterpret_cast<double2*>(T + 2 * rg.t);
  double2* Rr = Lr + G * nl2;
  const double sq = sqrt(p.dt);
  load_panel<NT>(b, w, P);
  load_trial<NT>(b, T);
  for (int s = 0; s < b.nbuf; ++s)
    for (int e = tid; e < NN; e += NT) E[s * NN + e] = p.ex[s][e];
  if (RES) {
#pragma unroll 8
    for (int e = tid; e < G * nl2; e += NT) Lr[e] = p.lt[e];
#pragma unroll 8
    for (int e = tid; e < G * nr2; e += NT) Rr[e] = p.rcp[e];
  }
  __syncthreads();
  overlap_matrices<NT>(b, T, P, S);
  __syncthreads();
  invert(b, S, det);
  __syncthreads();

  const Tiles<NT, TR, TPT> tl(N, c);
  double2 acc[TPT][TR][TR], term[TPT][TR][TR];
  // A (row stride lda) times the panel in, onto this thread's tiles
  auto times = [&](auto* A, int lda, int per_buf, const double2* in, double2 (&o)[TPT][TR][TR]) {
#pragma unroll
    for (int u = 0; u < TPT; ++u) {
#pragma unroll
      for (int i = 0; i < TR; ++i)
#pragma unroll
        for (int j = 0; j < TR; ++j) o[u][i][j] = double2{0.0, 0.0};
      if (!tl.on[u]) continue;
      const decltype(+A) ar[2] = {A + min(tl.row[u][0], N - 1) * lda, A + min(tl.row[u][TR - 1], N - 1) * lda};
      const int cc[2] = {min(tl.col[u][0], c - 1), min(tl.col[u][TR - 1], c - 1)};
      const int bo[2] = {cc[0] >= b.cb[0] ? per_buf : 0, cc[1] >= b.cb[0] ? per_buf : 0};
#pragma unroll 4
      for (int k = 0; k < N; ++k) {
        double2 bv[TR];
#pragma unroll
        for (int j = 0; j < TR; ++j) bv[j] = in[k * c + cc[j]];
#pragma unroll
        for (int i = 0; i < TR; ++i) {
          if constexpr (sizeof(*A) == sizeof(double)) {
#pragma unroll
            for (int j = 0; j < TR; ++j) {
              const double av = ar[i][bo[j] + k];
              o[u][i][j].x += av * bv[j].x;
              o[u][i][j].y += av * bv[j].y;
            }
          } else {
            const double2 av = ar[i][k];
#pragma unroll
            for (int j = 0; j < TR; ++j) {
              o[u][i][j].x = fma(av.x, bv[j].x, fma(-av.y, bv[j].y, o[u][i][j].x));
              o[u][i][j].y = fma(av.x, bv[j].y, fma(av.y, bv[j].x, o[u][i][j].y));
            }
          }
        }
      }
    }
  };
  auto put = [&](double2* out, const double2 (&o)[TPT][TR][TR]) {
#pragma unroll
    for (int u = 0; u < TPT; ++u)
#pragma unroll
      for (int i = 0; i < TR; ++i)
#pragma unroll
        for (int j = 0; j < TR; ++j)
          if (tl.on[u] && tl.row[u][i] < N && tl.col[u][j] < c) out[tl.row[u][i] * c + tl.col[u][j]] = o[u][i][j];
  };

  double2 oo = p.overlaps[w];
  for (int step = 0; step < p.nsteps; ++step) {
    const bool last = step + 1 == p.nsteps;
    const double* fields = p.fields + ((long)step * b.W + w) * G;
    greens<NT>(b, P, S, V);
    __syncthreads();

    // force bias and field shift: 16 lanes for each U Cholesky indices
    double2 sh = {0.0, 0.0}, ft = {0.0, 0.0};
    {
      constexpr int U = RES ? 1 : 5, EU = RES ? 2 : 3;
      const double2* R = RES ? Rr : p.rcp;
      const int grp = tid >> 4, l16 = tid & 15;
      for (int g0 = U * grp; g0 < G; g0 += U * (NT / 16)) {
        double2 f[U];
#pragma unroll
        for (int u = 0; u < U; ++u) f[u] = double2{0.0, 0.0};
        for (int e0 = l16; e0 < nr2; e0 += 16 * EU) {
          double2 rv[EU][U];
#pragma unroll
          for (int t = 0; t < EU; ++t)
#pragma unroll
            for (int u = 0; u < U; ++u) rv[t][u] = R[min(g0 + u, G - 1) * nr2 + min(e0 + 16 * t, nr2 - 1)];
#pragma unroll
          for (int t = 0; t < EU; ++t) {
            const int e = 2 * (e0 + 16 * t);
            const double2 ga = e < nrc ? V[e] : double2{0.0, 0.0}, gb = e + 1 < nrc ? V[e + 1] : double2{0.0, 0.0};
#pragma unroll
            for (int u = 0; u < U; ++u) {
              f[u].x += rv[t][u].x * ga.x + rv[t][u].y * gb.x;
              f[u].y += rv[t][u].x * ga.y + rv[t][u].y * gb.y;
            }
          }
        }
#pragma unroll
        for (int off = 8; off > 0; off >>= 1)
#pragma unroll
          for (int u = 0; u < U; ++u) {
            f[u].x += __shfl_xor(f[u].x, off);
            f[u].y += __shfl_xor(f[u].y, off);
          }
        if (l16 < U && g0 + l16 < G) {
          const int g = g0 + l16;
          double2 fb = f[0];
#pragma unroll
          for (int u = 1; u < U; ++u)
            if (l16 == u) fb = f[u];
          fb.x *= p.fac;
          fb.y *= p.fac;
          const double2 m = p.mf[g];
          const double xv = fields[g];
          const double2 s = {-sq * (-fb.y - m.x), -sq * (fb.x - m.y)};
          const double2 z = {xv - s.x, -s.y};
          const double2 ss = cmul(s, s);
          sh = cadd(sh, cmul(z, m));
          ft.x += xv * s.x - ss.x / 2.0;
          ft.y += xv * s.y - ss.y / 2.0;
          xs[g] = z;
          if (last) {
            p.xs[w * G + g] = z;
            p.fb[w * G + g] = fb;
          }
        }
      }
    }
    sh = group_sum2<NT>(sh, red);  // its barriers also end the reads of G in V
    ft = group_sum2<NT>(ft, red);

    // t0 = E W, and VHS = i sqrt(dt) sum_g xs_g L_g (mirrored where L_g is symmetric)
    times(E, N, NN, P, acc);
    put(Q, acc);
    {
      constexpr int GU = RES ? 4 : 16;
      const double2* L = RES ? Lr : p.lt;
      for (int e = tid; e < nl2; e += NT) {
        double2 v[2] = {{0.0, 0.0}, {0.0, 0.0}};
        for (int g = 0; g < G; g += GU) {
          double2 l[GU];
#pragma unroll
          for (int t = 0; t < GU; ++t) l[t] = L[min(g + t, G - 1) * nl2 + e];
#pragma unroll
          for (int t = 0; t < GU; ++t) {
            const double2 z = g + t < G ? xs[g + t] : double2{0.0, 0.0};
            v[0].x += z.x * l[t].x;
            v[0].y += z.y * l[t].x;
            v[1].x += z.x * l[t].y;
            v[1].y += z.y * l[t].y;
          }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          int i, j;
          vhs_entry(min(2 * e + u, nent - 1), N, p.sym, i, j);
          const double2 r = {-sq * v[u].y, sq * v[u].x};
          if (2 * e + u < nent) {
            V[i * rg.ldv + j] = r;
            if (p.sym) V[j * rg.ldv + i] = r;
          }
        }
      }
    }
    __syncthreads();

    double2* cur = Q;
    double2* nxt = P;
    for (int n = 1; n < p.nterms; ++n) {
      times(V, rg.ldv, 0, cur, term);
      const double f = 1.0 / n;
#pragma unroll
      for (int u = 0; u < TPT; ++u)
#pragma unroll
        for (int i = 0; i < TR; ++i)
#pragma unroll
          for (int j = 0; j < TR; ++j) {
            term[u][i][j].x *= f;
            term[u][i][j].y *= f;
            acc[u][i][j] = cadd(acc[u][i][j], term[u][i][j]);
          }
      if (n + 1 < p.nterms) {
        put(nxt, term);
        __syncthreads();
        double2* t = cur;
        cur = nxt;
        nxt = t;
      }
    }
    put(nxt, acc);
    __syncthreads();
    times(E, N, NN, nxt, acc);
    put(cur, acc);
    __syncthreads();
    P = cur;
    Q = nxt;
    overlap_matrices<NT>(b, T, P, S);
    __syncthreads();
    invert(b, S, det);
    __syncthreads();
    const double2 on = cmul(det[0], det[b.nspin - 1]);
    if (tid == NT - 1) {
      p.h[(long)step * b.W + w] = factor_call(on, oo, sh, ft, p.scalars[1], *p.h0p, p.dt);
      if (last) {
        p.overlaps[w] = on;
        p.terms[2 * w] = sh;
        p.terms[2 * w + 1] = ft;
        p.ov_new[w] = on;
      }
    }
    oo = on;
  }
  store_panel<NT>(b, w, P);
}

// The weights through nsteps steps: factor h exp(dt (shift - shift at the first
// step)), clipped (propagation.py:320-334), the shift following from each step's
// sum.  The factors are taken at the first step's shift and not at e_estimate,
// so that a step's weights do not depend on e_estimate (which may be far from
// the shift, or not finite) and a single step needs no rescaling.
__global__ __launch_bounds__(1024) void small_weights_kernel(const double* __restrict__ h, int nsteps, int W, double dt,
                                                             double* __restrict__ weights,
                                                             double* __restrict__ scalars) {
  __shared__ double red[2][16];
  const double e_est = scalars[0];
  const double first = scalars[1];
  double pcs = first;
  for (int s = 0; s < nsteps; ++s) {
    const double f = exp(dt * (pcs - first));
    double sum = 0.0;
    for (int w = threadIdx.x; w < W; w += 1024) {
      const double wn = wm::clipped_weight(f * h[(long)s * W + w], weights[w]);
      weights[w] = wn;
      sum += wn;
    }
    sum = wave_sum(sum);
    if ((threadIdx.x & 63) == 0) red[s & 1][threadIdx.x >> 6] = sum;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int i = 0; i < 16; ++i) t += red[s & 1][i];
    pcs = e_est - 0.1 * log(t / W) / dt;
  }
  if (threadIdx.x == 0) scalars[1] = pcs;
}

// Cholesky QR twice of every buffer's panel (at most 16 columns each), in place
// in X; R: one 16 x 16 triangle a buffer.
template <int NT>
__device__ inline void cholqr2(const SmallJob& b, double2* X, double2 (*R)[256]) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, N = b.N;
  const int c0 = b.cb[0], c1 = b.nbuf > 1 ? b.cb[1] : 0;
  for (int pass = 0; pass < 2; ++pass) {
    for (int e = tid; e < c0 * c0 + c1 * c1; e += NT) {
      const int s = e >= c0 * c0, cs = s ? c1 : c0, l = e - s * c0 * c0, i = l / cs, j = l - i * cs;
      const double2* x = X + (s ? c0 : 0);
      double2 a = {0.0, 0.0};
#pragma unroll 4
      for (int r = 0; r < N; ++r) {
        const double2 u = x[r * b.c + i], v = x[r * b.c + j];
        a.x += u.x * v.x + u.y * v.y;
        a.y += u.x * v.y - u.y * v.x;
      }
      R[s][l] = a;
    }
    __syncthreads();
    // upper factor in place, one wave a buffer
    if (wave < b.nbuf) {
      const int n = b.cb[wave];
      double2* A = R[wave];
      for (int k = 0; k < n; ++k) {
        const double d = sqrt(A[k * n + k].x), di = 1.0 / d;
        wm::wave_lds_sync();
        if (lane == 0) A[k * n + k] = double2{d, 0.0};
        if (lane > k && lane < n) {
          const double2 z = A[k * n + lane];
          A[k * n + lane] = double2{z.x * di, z.y * di};
        }
        wm::wave_lds_sync();
        for (int e = lane; e < n * n; e += 64) {
          const int i = e / n, j = e - i * n;
          if (i > k && j >= i) {
            const double2 u = A[k * n + i], v = A[k * n + j];
            A[e].x -= u.x * v.x + u.y * v.y;
            A[e].y -= u.x * v.y - u.y * v.x;
          }
        }
        wm::wave_lds_sync();
      }
    }
    __syncthreads();
    // rows of W R^-1: x_j = (w_j - sum_{i<j} x_i R_ij) / R_jj
    for (int t = tid; t < N * b.nbuf; t += NT) {
      const int s = t / N, r = t - s * N, n = b.cb[s];
      double2* x = X + r * b.c + (s ? c0 : 0);
      double2 v[16];
#pragma unroll
      for (int j = 0; j < 16; ++j)
        if (j < n) {
          double2 a = x[j];
#pragma unroll
          for (int i = 0; i < j; ++i) {
            const double2 u = R[s][i * n + j];
            a.x -= v[i].x * u.x - v[i].y * u.y;
            a.y -= v[i].x * u.y + v[i].y * u.x;
          }
          const double di = 1.0 / R[s][j * n + j].x;
          v[j] = double2{a.x * di, a.y * di};
          x[j] = v[j];
        }
    }
    __syncthreads();
  }
}

constexpr int kMeasureThreads = 256;

__global__ __launch_bounds__(kMeasureThreads) void small_measure_kernel(SmallMeasure p) {
  extern __shared__ double2 sm[];
  constexpr int NT = kMeasureThreads;
  __shared__ double2 S[2][256];
  __shared__ double2 det[2], red[NT / 64];
  const SmallJob& b = p.b;
  const int tid = threadIdx.x;
  const int N = b.N;
  const long w = blockIdx.x;
  const int osum = b.occ[0] + (b.nspin > 1 ? b.occ[1] : 0);
  double2* X = sm;             // the panel
  double2* V = X + N * b.c;    // the Green's functions
  double* T = reinterpret_cast<double*>(V + N * osum);
  load_panel<NT>(b, w, X);
  load_trial<NT>(b, T);
  __syncthreads();
  if (p.qr) {
    cholqr2<NT>(b, X, S);
    store_panel<NT>(b, w, X);
  }
  overlap_matrices<NT>(b, T, X, S);
  __syncthreads();
  invert(b, S, det);
  __syncthreads();
  if (tid == 0) {
    for (int s = 0; s < b.nspin; ++s) b.det[s][w] = det[s];
    if (p.overlaps) p.overlaps[w] = cmul(det[0], det[b.nspin - 1]);
  }
  if (!p.inverse) return;
  for (int s = 0; s < b.nspin; ++s) {
    const int n = b.occ[s] * b.occ[s];
    for (int e = tid; e < n; e += NT) b.Sinv[s][w * n + e] = S[s][e];
  }
  greens<NT>(b, X, S, V);
  __syncthreads();
  const double2* Gm = V;
  for (int s = 0; s < b.nspin; ++s) {
    const int n = b.occ[s] * N;
    for (int e = tid; e < n; e += NT) p.green[s][w * n + e] = Gm[e];
    Gm += n;
  }
  if (!p.energy) return;
  if (p.whole) {
    // E = h0 + tr(rot_h1 G^T) + 1/2 sum_g c_g^2 - 1/2 sum_g tr(f_g f_g), one
    // spin standing for both where nspin = 1; a thread forms f_ij and f_ji
    const double two = b.nspin == 1 ? 2.0 : 1.0;
    double2 e = {0.0, 0.0};
    Gm = V;
    for (int s = 0; s < b.nspin; ++s) {
      const int O = b.occ[s], n = O * N, OO = O * O;
      for (int t = tid; t < n; t += NT) {
        const double h = p.fac * p.rh1[s][t];
        e.x += h * Gm[t].x;
        e.y += h * Gm[t].y;
      }
      for (int t = tid; t < b.G * OO; t += NT) {
        const int g = t / OO, l = t - g * OO, i = l / O, j = l - i * O;
        const double *ri = p.rc[s] + (long)g * n + i * N, *rj = p.rc[s] + (long)g * n + j * N;
        const double2 *gi = Gm + i * N, *gj = Gm + j * N;
        double2 x = {0.0, 0.0}, y = {0.0, 0.0};
#pragma unroll 4
        for (int q = 0; q < N; ++q) {
          const double a = ri[q], c = rj[q];
          const double2 u = gj[q], v = gi[q];
          x.x += a * u.x;
          x.y += a * u.y;
          y.x += c * v.x;
          y.y += c * v.y;
        }
        const double2 k = cmul(x, y);
        e.x -= 0.5 * two * k.x;
        e.y -= 0.5 * two * k.y;
      }
      Gm += n;
    }
    for (int g = tid; g < b.G; g += NT) {
      double2 c = {0.0, 0.0};
      Gm = V;
      for (int s = 0; s < b.nspin; ++s) {
        const int n = b.occ[s] * N;
        const double* r = p.rc[s] + (long)g * n;
#pragma unroll 4
        for (int t = 0; t < n; ++t) {
          c.x += r[t] * Gm[t].x;
          c.y += r[t] * Gm[t].y;
        }
        Gm += n;
      }
      const double2 k = cmul(c, c);
      e.x += 0.5 * two * two * k.x;
      e.y += 0.5 * two * two * k.y;
    }
    e = group_sum2<NT>(e, red);
    if (tid == 0) p.energies[w] = double2{p.h0 + e.x, e.y};
    return;
  }
  double2 e1 = {0.0, 0.0};
  Gm = V;
  for (int s = 0; s < b.nspin; ++s) {
    const int O = b.occ[s], Nv = N - O, n = O * N;
    for (int e = tid; e < n; e += NT) {
      const double2 g = Gm[e];
      const double h = p.fac * p.rh1[s][e];
      e1.x += h * g.x;
      e1.y += h * g.y;
    }
    // theta_w (columns j) = Q^T G_w^T in the exchange's packed layout, zero
    // past Nv, and the walker's part of K that is linear in it
    if (!p.thetap[s]) {
      Gm += n;
      continue;
    }
    const int grp = (int)(w / p.wn[s]), wl = (int)(w - (long)grp * p.wn[s]), np2 = 2 * p.npr[s];
    double* out = reinterpret_cast<double*>(p.thetap[s]);
    double2 kk = {0.0, 0.0};
    for (int e = tid; e < O * np2; e += NT) {
      const int j = e / np2, k = e - j * np2;
      double2 t = {0.0, 0.0};
      if (k < Nv) {
        const double* q = p.q[s] + k;
        const double2* g = Gm + j * N;
#pragma unroll 4
        for (int r = 0; r < N; ++r) {
          const double qv = q[r * Nv];
          const double2 gv = g[r];
          t.x += qv * gv.x;
          t.y += qv * gv.y;
        }
        const double m = p.mt[s][j * Nv + k];
        kk.x += m * t.x;
        kk.y += m * t.y;
      }
      const long o = (((long)grp * p.npr[s] + (k >> 1)) * 2 * p.c2[s] + 2 * (wl * O + j)) * 2 + (k & 1);
      out[o] = t.x;
      out[o + 2] = t.y;
    }
    kk = group_sum2<NT>(kk, red);
    if (tid == 0)
      p.kpart[s][w * (p.nchunk[s] + 1) + p.nchunk[s]] = double2{*p.k0[s] + 2.0 * kk.x, 2.0 * kk.y};
    Gm += n;
  }
  e1 = group_sum2<NT>(e1, red);
  if (tid == 0) p.ene1[w] = e1;
}

__global__ void pack_l_kernel(const double* __restrict__ chol, int N, int G, int sym, int nent, int n2,
                              double2* __restrict__ out) {
  const long t = blockIdx.x * 256L + threadIdx.x;
  if (t >= (long)G * n2) return;
  const long g = t / n2;
  const int e = 2 * (int)(t - g * n2);
  const double* L = chol + g * N * N;
  int i, j;
  vhs_entry(e, N, sym, i, j);
  double2 v = {L[i * N + j], 0.0};
  if (e + 1 < nent) {
    vhs_entry(e + 1, N, sym, i, j);
    v.y = L[i * N + j];
  }
  out[t] = v;
}

__global__ void pack_rc_kernel(const double* __restrict__ rc0, int n0, const double* __restrict__ rc1, int n1, int G,
                               int n2, double2* __restrict__ out) {
  const long t = blockIdx.x * 256L + threadIdx.x;
  if (t >= (long)G * n2) return;
  const long g = t / n2;
  const int e = 2 * (int)(t - g * n2);
  auto at = [&](int i) { return i < n0 ? rc0[g * n0 + i] : i - n0 < n1 ? rc1[g * n1 + i - n0] : 0.0; };
  out[t] = double2{at(e), at(e + 1)};
}

// Dynamic LDS at most: of a step that streams L and rot_chol, of one that holds
// them (two work-groups a CU), and of a measurement.
constexpr size_t kStepLds = 144 * 1024, kResidentLds = 72 * 1024, kMeasureLds = 96 * 1024;

int osum_of(const SmallJob& b) { return b.occ[0] + (b.nspin > 1 ? b.occ[1] : 0); }

template <int NT, int TR, int TPT, bool RES>
int launch_step(const SmallStep& p, size_t bytes, hipStream_t st) {
  static std::atomic<uint64_t> raised{0};
  AFQ_TRY(raise_lds(reinterpret_cast<const void*>(small_step_kernel<NT, TR, TPT, RES>),
                    RES ? kResidentLds : kStepLds, raised, "small step"));
  hipLaunchKernelGGL((small_step_kernel<NT, TR, TPT, RES>), dim3(p.b.W), dim3(NT), bytes, st, p);
  return launch_status("small_step_kernel");
}

}  // namespace

size_t small_step_lds(int N, int G, int c, int osum, int nbuf) {
  if (N > kSmallMaxN || G > 2048) return 0;
  const Regions r = regions(N, c, osum, nbuf);
  const size_t bytes = sizeof(double2) * (2 * r.panel + r.v + r.e + r.t + G);
  return bytes <= kStepLds ? bytes : 0;
}

// A thread then forms at most some 400 products of the exchange, fewer than the
// launches it replaces take (N = 12, O = 3 / 2, G = 40, 200 walkers: 41.5 us an
// energy with the exchange kernel, 15.6 us here; N = 20, O = 7, G = 50, 512
// walkers 29.9 us against 55.6 before either).
bool small_energy_whole(int N, int G, int occ0, int occ1) {
  return (long)G * N * (occ0 * occ0 + occ1 * occ1) <= 50000;
}

// One spin up to N osum = 1536, two spins, which save twice the launches, to 2400
// (the LDS): an energy here and by separate launches, N = 120, O = 16, G = 400,
// N osum = 1920: 1 walker 56 and 54 us, 32 walkers 107 and 103, 2048 walkers 3.08
// and 2.73 ms; UHF N = 60, O = 14 / 13, G = 300, 1620: 52 and 68 us, 76 and 79, 1.42
// and 1.52 ms; UHF N = 76, O = 16 / 15, G = 400, 2356: 55 and 68, 125 and 123, 4.12
// and 4.17.
size_t small_measure_lds(int N, int c, int osum, int nspin) {
  const size_t bytes = sizeof(double2) * (size_t)N * (c + osum) + sizeof(double) * (size_t)N * osum;
  return N * osum <= (nspin > 1 ? 2400 : 1536) && bytes <= kMeasureLds ? bytes : 0;
}

long small_l_pairs(int N, bool sym) { return (vhs_entries(N, sym) + 1) / 2; }
long small_rc_pairs(int N, int osum) { return (N * osum + 1) / 2; }

int k_small_pack_l(const double* chol, int N, int G, bool sym, double2* out, hipStream_t st) {
  const long n2 = small_l_pairs(N, sym), n = G * n2;
  hipLaunchKernelGGL(pack_l_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, chol, N, G, sym ? 1 : 0,
                     vhs_entries(N, sym), (int)n2, out);
  return launch_status("pack_l_kernel");
}

int k_small_pack_rc(const double* rc0, int n0, const double* rc1, int n1, int G, double2* out, hipStream_t st) {
  const long n2 = (n0 + n1 + 1) / 2, n = G * n2;
  hipLaunchKernelGGL(pack_rc_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, rc0, n0, rc1, n1, G, (int)n2,
                     out);
  return launch_status("pack_rc_kernel");
}

// The bytes of L and rot_chol a CU reads for its walkers (work-groups over 256 CUs)
// against the launches saved.  Where L is packed (sym), the launches are those of the
// fused propagator, and the line lies at about 2.5 MB a CU (UHF, separate and here):
//   N = 48, O = 9 / 9:    G = 60, 256 walkers (1.0 MB) 116 / 81 us; 512 (2.0) 155 / 147;
//                         1024 (3.9) 255 / 278; G = 115, 257 (3.8) 161 / 158;
//   N = 48, O = 16 / 16:  G = 115, 4 walkers (2.5 MB) 106 / 117, 256 149 / 125, 257
//                         (5.0) 197 / 228; G = 160, 64 (3.5) 130 / 129, 512 (6.9) 216 / 250.
// Where it is not, each product is a launch of the general kernel, and it lies near
// 10 MB:
//   N = 20, O = 6 / 6:    G = 450, 256 walkers (2.3 MB) 183 / 75, 1024 (9.2) 261 / 165;
//   N = 30, O = 8 / 8:    G = 300, 256 (3.3) 168 / 88; G = 450, 257 (9.9) 198 / 195;
//                         G = 300, 1024 (13.2) 278 / 299;
//   N = 40, O = 10 / 10:  G = 300, 256 (5.8) 209 / 124; G = 300, 257 (11.5) 234 / 229.
bool small_step_pays(int N, int G, int osum, int W, bool sym) {
  const double bytes = 8.0 * G * (vhs_entries(N, sym) + N * osum);
  return bytes * ((W + 255) / 256) <= (sym ? 2.5e6 : 9.5e6);
}

int k_small_step(const SmallStep& p, hipStream_t st) {
  const SmallJob& b = p.b;
  const int osum = osum_of(b);
  const size_t bytes = small_step_lds(b.N, b.G, b.c, osum, b.nbuf);
  if (bytes == 0) return fail(AFQ_E_UNSUPPORTED, "small step: sizes past the limits");
  const size_t res = bytes + sizeof(double2) * (size_t)b.G * (small_l_pairs(b.N, p.sym) + small_rc_pairs(b.N, osum));
  if (b.N * b.c <= 256) {
    if (res <= kResidentLds) return launch_step<256, 1, 1, true>(p, res, st);
    return launch_step<256, 1, 1, false>(p, bytes, st);
  }
  if (res <= kResidentLds) return launch_step<512, 1, 3, true>(p, res, st);
  return launch_step<512, 2, 1, false>(p, bytes, st);
}

int k_small_weights(const double* h, int nsteps, int W, double dt, double* weights, double* scalars, hipStream_t st) {
  hipLaunchKernelGGL(small_weights_kernel, dim3(1), dim3(1024), 0, st, h, nsteps, W, dt, weights, scalars);
  return launch_status("small_weights_kernel");
}

int k_small_measure(const SmallMeasure& p, hipStream_t st) {
  const size_t bytes = small_measure_lds(p.b.N, p.b.c, osum_of(p.b), p.b.nspin);
  if (bytes == 0) return fail(AFQ_E_UNSUPPORTED, "small measurement: sizes past the limits");
  static std::atomic<uint64_t> raised{0};
  AFQ_TRY(raise_lds(reinterpret_cast<const void*>(small_measure_kernel), kMeasureLds, raised, "small measurement"));
  hipLaunchKernelGGL(small_measure_kernel, dim3(p.b.W), dim3(kMeasureThreads), bytes, st, p);
  return launch_status("small_measure_kernel");
}

}  // namespace afq

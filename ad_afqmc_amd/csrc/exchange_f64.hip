// FP64 Coulomb/exchange measurement over the unoccupied orbitals of the trial.
//
// For walker w and Cholesky index g: f_g = rot_chol_g (O x N) . G_w^T (N x O),
// c_g = tr f_g, K = sum_g sum_ij f_g,ij f_g,ji (ad_afqmc/wavefunctions.py:1137-1139,
// 1347-1356).  T^T G_w^T = 1 for every walker (G_w^T = W (T^T W)^-1), so with an
// orthonormal basis Q of the complement of span(T) (N x Nv, Nv = N - O) and
// P = T (T^T T)^-1
//     G_w^T = P + Q theta_w,   theta_w = Q^T G_w^T   (Nv x O),
//     f_g   = f0_g + d_g,      f0_g = rot_chol_g P,  d_g = (rot_chol_g Q) theta_w.
// f0 does not depend on the walker, so its part of K collapses to a constant
// and one matrix M (O x Nv):
//     c_g = tr f0_g + tr d_g
//     K   = sum_g tr(f0_g f0_g) + 2 sum_ja M_ja theta_aj + sum_g tr(d_g d_g),
//     M   = sum_g f0_g (rot_chol_g Q).
// Only tr d_g and tr(d_g d_g) cost O(G O^2 Nv) per walker; the contraction runs
// over N - O instead of N orbitals.  f0, M and rot_chol_g Q are built once per
// (rot_chol, trial).
//
// d as one product.  The rows (g, i) of gw consecutive g are stacked without
// gaps, and so are the columns (walker, j, re/im) of wn walkers, so 16 x 16
// MFMA blocks are padded once per tile and not once per f block: O = 40 fills
// 120 of 128 rows and 80 of 80 columns (48 x 48 per f block before: 1.44 times
// the work).  A work-group of WR x WC waves holds the tile's d in registers,
// MB x NB blocks a wave.  A (rot_chol Q) goes straight from global memory to
// registers (no other wave of the row needs it; 1 KB of consecutive bytes per
// fragment pair, fetched one 8-deep step ahead), B (theta) is staged in LDS in
// 16-deep slabs as pairs of consecutive k, so one 16-byte read feeds two
// MFMAs; the next slab is in flight while the current one is multiplied.
// Then d goes through LDS, where every d_ij meets its d_ji.
//
// Bound: the FP64 matrix cores (4 G O^2 Nv flops a walker, 85% of the rate a
// large FP64 product reaches at O = 60 counting the tile's padding; the rest is
// the passes of d through LDS).  Measured against the kernels before (f over all
// N orbitals, one wave per f block): N = 200, O = 40, G = 1200, 512 walkers
// 17.7 -> 12.2 ms a measurement; N = 300, O = 60 / 58, G = 2000, 256 walkers
// 110.5 -> 67.1 ms; N = 250, O = 82, G = 1010, 48 walkers (f stored in memory
// before) 14.2 -> 6.1 ms, with the inverse in registers.
#include "exchange_f64.h"

#include "kernels.h"

namespace afq {
namespace {

__device__ inline double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

constexpr int kSteps = 4;             // 8-deep steps of a slab of B
constexpr int kPairs = 4 * kSteps;    // its k pairs

// Register budget: three waves a SIMD where the accumulators leave room.
constexpr int waves_per_simd(int mb, int nb, int waves) { return waves == 4 && mb * nb <= 10 ? 3 : 2; }
// LDS bytes for the passes of d: as many work-groups a CU as the registers allow.
constexpr size_t tile_room(int mb, int nb, int waves) {
  const int per_cu = waves_per_simd(mb, nb, waves) * 4 / waves;
  return (per_cu == 3 ? 46 : per_cu == 2 ? 74 : 148) * 1024;
}

template <int MB, int NB, int WR, int WC>
__global__ __launch_bounds__(64 * WR * WC, (waves_per_simd(MB, NB, WR * WC))) void exchange_f64_kernel(ExF64 p) {
  constexpr int NT = 64 * WR * WC;
  constexpr int RB = MB * WR;        // row blocks of the tile
  constexpr int C = 16 * NB * WC;    // columns of the tile
  extern __shared__ double2 lds[];   // [2][kPairs][C] slabs, then d of one g
  __shared__ double2 trace;
  __shared__ double2 ksum[NT];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave / WC, wc = wave % WC;
  const int q = lane >> 4, c16 = lane & 15;
  const int O = p.O, Nv = p.Nv;

  // XCD-aware order: XCD x takes a contiguous range of (chunk group, walkers,
  // chunk in group), so a group's slice of A stays in its L2
  const long L = (long)(blockIdx.x & 7) * p.T8 + (blockIdx.x >> 3);
  const long per_group = (long)p.nwg * p.cpg;
  const long grp = L / per_group;
  const long rem = L - grp * per_group;
  const int w0 = (int)(rem / p.cpg) * p.wn;
  const int chunk = (int)(grp * p.cpg + rem % p.cpg);
  if (chunk >= p.nchunk) return;  // uniform for the work-group
  const int nw = min(p.wn, p.W - w0);

  v4d acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};

  const int n8 = p.n8;
  if (n8 > 0) {
    // B: packed slabs in the LDS layout, copied by the DMA path, wave by wave
    // in pieces of 64 x 16 bytes
    constexpr int SLAB = kPairs * C, PIECES = SLAB / 64, PPW = (PIECES + WR * WC - 1) / (WR * WC);
    const int nslab = (n8 + kSteps - 1) / kSteps;
    const double2* src = p.theta + (long)(w0 / p.wn) * nslab * SLAB + lane;
    auto copy = [&](int slab, int buf) {
#pragma unroll
      for (int t = 0; t < PPW; ++t) {
        const int piece = t * WR * WC + wave;
        if (PIECES % (WR * WC) == 0 || piece < PIECES)
          __builtin_amdgcn_global_load_lds(static_cast<const void*>(src + (long)slab * SLAB + 64 * piece),
                                           (__attribute__((address_space(3))) void*)(lds + buf * SLAB + 64 * piece),
                                           16, 0, 0);
      }
    };
    const double2* A = reinterpret_cast<const double2*>(p.a) + ((long)chunk * RB + wr * MB) * n8 * 64 + lane;
    double2 a[MB], an[MB], b[NB];
    copy(0, 0);
#pragma unroll
    for (int i = 0; i < MB; ++i) a[i] = A[(long)i * n8 * 64];
    for (int s = 0; s < nslab; ++s) {
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's copies have landed
      __syncthreads();
      if (s + 1 < nslab) copy(s + 1, (s + 1) & 1);
      const double2* B = lds + (s & 1) * SLAB + q * C + wc * NB * 16 + c16;
      const int nt = min(kSteps, n8 - kSteps * s);
#pragma unroll
      for (int t = 0; t < kSteps; ++t) {
        if (t >= nt) break;  // uniform
        const int kn = min(kSteps * s + t + 1, n8 - 1);
#pragma unroll
        for (int i = 0; i < MB; ++i) an[i] = A[((long)i * n8 + kn) * 64];
#pragma unroll
        for (int j = 0; j < NB; ++j) b[j] = B[4 * t * C + 16 * j];
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].x, b[j].x, acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].y, b[j].y, acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < MB; ++i) a[i] = an[i];
      }
    }
    __syncthreads();
  }

  // d through LDS, pass by pass: rows [r0, r1) of the tile (p.gp whole g's, or
  // p.strip rows of one g where a g does not fit) as F[row - r0][column], row
  // stride LD = 2 (mod 16) doubles, so that rows read down a column start in
  // distinct 16-byte banks.  A strip also needs its columns of every row of
  // the g (Y).  Element v of block (i, j) is row 16 (wr MB + i) + q + 4 v,
  // column 16 (wc NB + j) + c16.
  constexpr int LD = C + 2;
  double* F = reinterpret_cast<double*>(lds);
  const int gcnt = min(p.gw, p.G - chunk * p.gw);
  const bool strips = p.strip < O;
  const int LDY = strips ? 2 * p.strip + 2 : LD;
  double* Y = strips ? F + p.strip * LD : F;
  const int rstep = strips ? p.strip : p.gp * O;
  // threads of walker wl: tw consecutive ones
  const int tw = NT / nw, wl = tid / tw, sub = tid - wl * tw;
  const float invO = 1.0f / O;
  double kr = 0.0, ki = 0.0;
  for (int r0 = 0; r0 < gcnt * O; r0 += rstep) {
    const int r1 = min(gcnt * O, r0 + rstep);
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = 16 * (wr * MB + i) + q + 4 * v;
        if (r >= r0 && r < r1) {
#pragma unroll
          for (int j = 0; j < NB; ++j) F[(r - r0) * LD + 16 * (wc * NB + j) + c16] = acc[i][j][v];
        }
        if (strips && r < O) {
#pragma unroll
          for (int j = 0; j < NB; ++j) {
            const int col = 16 * (wc * NB + j) + c16 - 2 * r0;
            if (col >= 0 && col < 2 * (r1 - r0)) Y[r * LDY + col] = acc[i][j][v];
          }
        }
      }
    __syncthreads();
    // sum over (row, j) of d_ij d_ji, four pairs in flight
    if (wl < nw) {
      const int n = (r1 - r0) * O;
      for (int e0 = sub; e0 < n; e0 += 4 * tw) {
        double2 x[4], y[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int e = min(e0 + u * tw, n - 1);
          const int lr = (int)((e + 0.5f) * invO), j = e - lr * O;
          const int gb = strips ? 0 : (int)((lr + 0.5f) * invO) * O;  // first row of the g
          x[u] = *reinterpret_cast<const double2*>(F + lr * LD + 2 * (wl * O + j));
          y[u] = *reinterpret_cast<const double2*>(Y + (gb + j) * LDY + 2 * (wl * O + lr - gb));
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (e0 + u * tw >= n) y[u] = double2{0.0, 0.0};
          kr += x[u].x * y[u].x - x[u].y * y[u].y;
          ki += x[u].x * y[u].y + x[u].y * y[u].x;
        }
      }
    }
    // traces: lt consecutive lanes for each (g, walker)
    const int ng = strips ? 1 : (r1 - r0) / O, len = strips ? r1 - r0 : O;
    const int lt = O > 32 ? 16 : O > 8 ? 4 : 1, l0 = lane & (lt - 1);
    for (int t = tid / lt; t < ng * nw; t += NT / lt) {
      const int gl = t / nw, wt = t - gl * nw;
      double cr = 0.0, ci = 0.0;
      for (int i = l0; i < len; i += lt) {
        const double2 z = *reinterpret_cast<const double2*>(F + (gl * O + i) * LD + 2 * (wt * O + i + (strips ? r0 : 0)));
        cr += z.x;
        ci += z.y;
      }
      for (int off = lt >> 1; off > 0; off >>= 1) {
        cr += __shfl_xor(cr, off);
        ci += __shfl_xor(ci, off);
      }
      if (l0 == 0) {
        if (strips) {
          if (r0 > 0) {
            cr += trace.x;
            ci += trace.y;
          }
          trace = double2{cr, ci};
        }
        if (!strips || r1 == O) {
          const int g = chunk * p.gw + (strips ? 0 : r0 / O) + gl;
          p.coul[(long)(w0 + wt) * p.G + g] = double2{p.c0[g] + cr, ci};
        }
      }
    }
    __syncthreads();
  }
  ksum[tid] = double2{kr, ki};
  __syncthreads();
  for (int w = wave; w < nw; w += WR * WC) {
    double sr = 0.0, si = 0.0;
    for (int e = lane; e < tw; e += 64) {
      sr += ksum[w * tw + e].x;
      si += ksum[w * tw + e].y;
    }
    sr = wave_sum(sr);
    si = wave_sum(si);
    if (lane == 0) p.kpart[(long)(w0 + w) * p.kstride + chunk] = double2{sr, si};
  }
}

// theta^T (W, O, Nv) -> per group of wn walkers the slabs of B: [slab][k pair]
// [column (walker, j, re/im)][2], zero past Nv, past the columns and past W.
// Consecutive threads take consecutive k pairs of one (walker, j).
__global__ void pack_b_kernel(const double2* __restrict__ theta, int O, int Nv, int wn, int W, int C2, int nslab,
                              long n, double2* __restrict__ out) {
  const long e = blockIdx.x * 256L + threadIdx.x;
  if (e >= n) return;
  const int npr = nslab * kPairs;
  const int pr = (int)(e % npr);
  const long r = e / npr;
  const int cj = (int)(r % C2);
  const long grp = r / C2;
  const int wl = cj / O;
  const long w = grp * wn + wl;
  const int k = 2 * pr;
  double2 x = {0.0, 0.0}, y = {0.0, 0.0};
  if (wl < wn && w < W) {
    const double2* t = theta + (w * O + (cj - wl * O)) * (long)Nv;
    if (k < Nv) x = t[k];
    if (k + 1 < Nv) y = t[k + 1];
  }
  double2* o = out + (grp * npr + pr) * 2L * C2 + 2 * cj;
  o[0] = double2{x.x, y.x};
  o[1] = double2{x.y, y.y};
}

long exchange_thetap_elems(const ExF64Tile& t, int Nv, int W) {
  const int nslab = ((Nv + 7) / 8 + kSteps - 1) / kSteps;
  return (long)((W + t.wn - 1) / t.wn) * nslab * kPairs * 16 * t.NB * t.WC;
}

// The same for few walkers, straight from their Green's functions, in one launch
// for both spins: theta_w of rows j0 .. j0 + 3 and 64 k's, each wave an eighth of
// the sum over the orbitals, and these elements' part of 2 sum_ja M_ja theta_aj
// (with K0, the first one's) in a slot of its own; and the one-body energies, a
// work-group a walker.  Zero past Nv; columns of walkers past W stay unread.
// Bound: the reads of Q, which each walker repeats (exchange_f64_few).
constexpr int kThetaRows = 4, kThetaWaves = 8;
struct ThetaSet {
  const double2* green;
  const double *Q, *mt, *k0, *rh1;
  int O, nx, wn, C2, npr, nchunk, kstride;  // nx: blocks of 64 k's
  double2* out;
  double2* kpart;
};
struct ThetaArgs {
  ThetaSet s[2];
  int nsets, N;
  double fac;
  double2* ene1;
};
__global__ __launch_bounds__(64 * kThetaWaves) void theta_kernel(ThetaArgs a) {
  __shared__ double2 part[kThetaWaves][kThetaRows][64];
  __shared__ double2 red[kThetaWaves];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int N = a.N;
  const long w = blockIdx.z;
  int x = blockIdx.x;
  if (x == a.s[0].nx + a.s[1].nx) {
    if (blockIdx.y > 0) return;
    double er = 0.0, ei = 0.0;
    for (int s = 0; s < a.nsets; ++s) {
      const int n = a.s[s].O * N;
      const double2* g = a.s[s].green + w * n;
      for (int e = threadIdx.x; e < n; e += 64 * kThetaWaves) {
        const double h = a.fac * a.s[s].rh1[e];
        er += h * g[e].x;
        ei += h * g[e].y;
      }
    }
    er = wave_sum(er);
    ei = wave_sum(ei);
    if (lane == 0) red[wave] = double2{er, ei};
    __syncthreads();
    if (threadIdx.x == 0) {
      double2 s = red[0];
      for (int i = 1; i < kThetaWaves; ++i) {
        s.x += red[i].x;
        s.y += red[i].y;
      }
      a.ene1[w] = s;
    }
    return;
  }
  const bool second = x >= a.s[0].nx;
  const ThetaSet& p = a.s[second ? 1 : 0];
  if (second) x -= a.s[0].nx;
  const int j0 = kThetaRows * blockIdx.y, k = 64 * x + lane, Nv = N - p.O;
  if (j0 >= p.O) return;
  const int rs = (N + kThetaWaves - 1) / kThetaWaves, r0 = min(N, wave * rs), r1 = min(N, r0 + rs);
  const double* q = p.Q + min(k, Nv - 1);
  const double2* g[kThetaRows];
  double2 acc[kThetaRows];
#pragma unroll
  for (int j = 0; j < kThetaRows; ++j) {
    g[j] = p.green + (w * p.O + min(j0 + j, p.O - 1)) * N;
    acc[j] = double2{0.0, 0.0};
  }
#pragma unroll 8
  for (int r = r0; r < r1; ++r) {
    const double b = q[(long)r * Nv];
#pragma unroll
    for (int j = 0; j < kThetaRows; ++j) {
      const double2 z = g[j][r];
      acc[j].x += b * z.x;
      acc[j].y += b * z.y;
    }
  }
#pragma unroll
  for (int j = 0; j < kThetaRows; ++j) part[wave][j][lane] = acc[j];
  __syncthreads();
  static_assert(kThetaRows <= kThetaWaves, "a wave finishes a row");
  const int j = j0 + wave;
  double2 t = {0.0, 0.0};
  if (wave < kThetaRows && k < Nv) {
#pragma unroll
    for (int i = 0; i < kThetaWaves; ++i) {
      t.x += part[i][wave][lane].x;
      t.y += part[i][wave][lane].y;
    }
  }
  double sr = 0.0, si = 0.0;
  if (wave < kThetaRows && j < p.O && k < 2 * p.npr) {
    const long grp = w / p.wn;
    double* o = reinterpret_cast<double*>(p.out) +
                (((grp * p.npr + (k >> 1)) * 2 * p.C2 + 2 * ((w - grp * p.wn) * p.O + j)) * 2 + (k & 1));
    o[0] = t.x;
    o[2] = t.y;
    if (k < Nv) {
      const double m = p.mt[(long)j * Nv + k];
      sr = m * t.x;
      si = m * t.y;
    }
  }
  sr = wave_sum(sr);
  si = wave_sum(si);
  if (lane == 0) red[wave] = double2{sr, si};
  __syncthreads();
  if (threadIdx.x == 0) {
    double2 s = {0.0, 0.0};
    for (int i = 0; i < kThetaRows; ++i) {
      s.x += red[i].x;
      s.y += red[i].y;
    }
    const int slot = blockIdx.y * p.nx + x;
    p.kpart[w * p.kstride + p.nchunk + slot] = double2{2.0 * s.x + (slot == 0 ? *p.k0 : 0.0), 2.0 * s.y};
  }
}

// kpart[w][nchunk] = K0 + 2 sum_ja M_ja theta_w,aj
__global__ __launch_bounds__(256) void exchange_occ_kernel(const double2* __restrict__ theta,
                                                           const double* __restrict__ mt,
                                                           const double* __restrict__ k0, long n, int nchunk,
                                                           double2* __restrict__ kpart) {
  __shared__ double2 red[4];
  const long w = blockIdx.x;
  const double2* th = theta + w * n;
  double sr = 0.0, si = 0.0;
  for (long e = threadIdx.x; e < n; e += 256) {
    const double2 t = th[e];
    sr += mt[e] * t.x;
    si += mt[e] * t.y;
  }
  sr = wave_sum(sr);
  si = wave_sum(si);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = double2{sr, si};
  __syncthreads();
  if (threadIdx.x == 0) {
    double2 s = {0.0, 0.0};
    for (int i = 0; i < 4; ++i) {
      s.x += red[i].x;
      s.y += red[i].y;
    }
    kpart[w * (nchunk + 1) + nchunk] = double2{*k0 + 2.0 * s.x, 2.0 * s.y};
  }
}

// ------------------------------------------------------------------ setup
// QR factors of the trial orbitals T = Q1 R (both spins in a launch, blockIdx.y):
// Q completes Q1 to an orthogonal matrix, and P = T (T^T T)^-1 = Q1 R^-T.  Taken
// from R, P is off by the condition of T.  By way of the Gram matrix T^T T, whose
// condition is its square, the energies of trials with condition 1e3 to 1e5 were
// off by 1.6 times what f = rot_chol G^T itself gives in FP64; by 0.74 times now.
struct TrialQR {
  const double* T;  // (N, O)
  int O;
  double* V;        // (O, N) Householder vectors
  double* tau;      // (O,)
  double* RT;       // (O, O) R by columns, upper part
  double* Q1;       // (N, O)
  double* Q;        // (N, N - O)
  double* P;        // (N, O)
};
struct TrialQR2 {
  TrialQR s[2];
};

// Column k's reflector is H_k = 1 - tau_k v_k v_k^T with v_k zero above row k.
// One work-group; a wave updates whole columns, in LDS where they fit (LOC).
template <bool LOC>
__global__ __launch_bounds__(1024) void householder_kernel(TrialQR2 sets, int N) {
  extern __shared__ double hv[];
  __shared__ double stau;
  const TrialQR& q = sets.s[blockIdx.y];
  const int O = q.O;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double* X = LOC ? hv : q.V;
  for (long e = tid; e < (long)N * O; e += 1024) X[(e % O) * N + e / O] = q.T[e];
  __syncthreads();
  for (int k = 0; k < O; ++k) {
    double* v = X + (long)k * N;
    if (wave == 0) {
      double s = 0.0;
      for (int r = k + lane; r < N; r += 64) s += v[r] * v[r];
      s = wave_sum(s);
      const double x = v[k], nrm = sqrt(s);
      const double vk = x + (x < 0.0 ? -nrm : nrm);
      // v^T v = s - x^2 + vk^2 = 2 nrm (nrm + |x|)
      const double vv = 2.0 * nrm * (nrm + fabs(x));
      const double t = vv > 0.0 ? 2.0 / vv : 0.0;
      for (int r = lane; r < k; r += 64) {
        q.RT[k * O + r] = v[r];
        v[r] = 0.0;
      }
      if (lane == 0) {
        q.RT[k * O + k] = x < 0.0 ? nrm : -nrm;
        v[k] = vk;
        q.tau[k] = t;
        stau = t;
      }
    }
    __syncthreads();
    const double t = stau;
    for (int j = k + 1 + wave; j < O; j += 16) {
      double* a = X + (long)j * N;
      double d = 0.0;
      for (int r = k + lane; r < N; r += 64) d += v[r] * a[r];
      d = t * wave_sum(d);
      for (int r = k + lane; r < N; r += 64) a[r] -= d * v[r];
    }
    __syncthreads();
  }
  if (LOC)
    for (long e = tid; e < (long)N * O; e += 1024) q.V[e] = X[e];
}

// Column blockIdx.x of H_0 ... H_{O-1}: the first O are Q1, the others Q.  One
// wave each, a lane owning the rows lane + 64 t: R of them in registers, or in
// memory where R = 0.
template <int R>
__global__ __launch_bounds__(64) void basis_kernel(TrialQR2 sets, int N) {
  const TrialQR& q = sets.s[blockIdx.y];
  const int a = blockIdx.x, lane = threadIdx.x, O = q.O;
  const int ld = a < O ? O : N - O;
  double* x = a < O ? q.Q1 + a : q.Q + (a - O);
  if constexpr (R > 0) {
    double y[R];
#pragma unroll
    for (int t = 0; t < R; ++t) y[t] = lane + 64 * t == a ? 1.0 : 0.0;
    for (int k = O - 1; k >= 0; --k) {
      double v[R], d = 0.0;
#pragma unroll
      for (int t = 0; t < R; ++t) v[t] = lane + 64 * t < N ? q.V[(long)k * N + lane + 64 * t] : 0.0;  // 0 above k
#pragma unroll
      for (int t = 0; t < R; ++t) d += v[t] * y[t];
      d = q.tau[k] * wave_sum(d);
#pragma unroll
      for (int t = 0; t < R; ++t) y[t] -= d * v[t];
    }
#pragma unroll
    for (int t = 0; t < R; ++t)
      if (lane + 64 * t < N) x[(long)(lane + 64 * t) * ld] = y[t];
    return;
  }
  for (int r = lane; r < N; r += 64) x[(long)r * ld] = r == a ? 1.0 : 0.0;
  for (int k = O - 1; k >= 0; --k) {
    const double* v = q.V + (long)k * N;
    const int r0 = k + ((lane - k) & 63);
    double d = 0.0;
    for (int r = r0; r < N; r += 64) d += v[r] * x[(long)r * ld];
    d = q.tau[k] * wave_sum(d);
    for (int r = r0; r < N; r += 64) x[(long)r * ld] -= d * v[r];
  }
}

// Row r of P = Q1 R^-T: R p = (row r of Q1), by back substitution.  One wave a
// row, lane i holding the entries i and i + 64.
__global__ __launch_bounds__(64) void dual_kernel(TrialQR2 sets) {
  static_assert(kExchangeF64MaxO <= 128, "two entries a lane");
  const TrialQR& q = sets.s[blockIdx.y];
  const int lane = threadIdx.x, O = q.O;
  const long row = (long)blockIdx.x * O;
  double x[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) x[h] = lane + 64 * h < O ? q.Q1[row + lane + 64 * h] : 0.0;
  for (int j = O - 1; j >= 0; --j) {
    const double* c = q.RT + (long)j * O;
    const double pj = __shfl(j < 64 ? x[0] : x[1], j & 63) / c[j];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int i = lane + 64 * h;
      const double ci = i < j ? c[i] : 0.0;
      x[h] = i == j ? pj : i < j ? x[h] - ci * pj : x[h];
    }
  }
#pragma unroll
  for (int h = 0; h < 2; ++h)
    if (lane + 64 * h < O) q.P[row + lane + 64 * h] = x[h];
}

// Tile rows of A from rcv (gn x O x Nv, chunks [0, nck) of gw g's): per chunk,
// RB row blocks of n8 8-deep steps of [k pair q][row][2], zero past the chunk's
// rows, past gn and past Nv.
__global__ void pack_a_kernel(const double* __restrict__ rcv, int O, int Nv, int gw, int gn, int RB, int n8, long nck,
                              double2* __restrict__ out) {
  const long per = (long)RB * n8 * 64;
  const long e = blockIdx.x * 256L + threadIdx.x;
  if (e >= nck * per) return;
  const long ck = e / per;
  const int t = (int)(e - ck * per);
  const int l = t & 63, s = (t >> 6) % n8, rb = (t >> 6) / n8;
  const int row = 16 * rb + (l & 15), k = 8 * s + 2 * (l >> 4);
  const long g = ck * gw + row / O;
  double2 v = {0.0, 0.0};
  if (row < gw * O && g < gn) {
    const double* r = rcv + (g * O + row % O) * (long)Nv;
    if (k < Nv) v.x = r[k];
    if (k + 1 < Nv) v.y = r[k + 1];
  }
  out[e] = v;
}

// f (gn, O, O): c0[g] = tr f_g, kg[g] = tr(f_g f_g), ft_g = f_g^T
__global__ __launch_bounds__(256) void occ_terms_kernel(const double* __restrict__ f, int O, double* __restrict__ c0,
                                                        double* __restrict__ kg, double* __restrict__ ft) {
  __shared__ double red[8];
  const long g = blockIdx.x;
  const double* fg = f + g * O * O;
  double c = 0.0, k = 0.0;
  for (int e = threadIdx.x; e < O * O; e += 256) {
    const int i = e / O, j = e - i * O;
    const double x = fg[e], y = fg[j * O + i];
    k += x * y;
    if (i == j) c += x;
    ft[g * O * O + e] = y;
  }
  c = wave_sum(c);
  k = wave_sum(k);
  if ((threadIdx.x & 63) == 0) {
    red[threadIdx.x >> 6] = c;
    red[4 + (threadIdx.x >> 6)] = k;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    c0[g] = red[0] + red[1] + red[2] + red[3];
    kg[g] = red[4] + red[5] + red[6] + red[7];
  }
}

// Sums of the set-up: mt[e] = sum_i part[i][e] over ns slices of n, and k0 = sum_g
// kg[g] (the last work-group); 16 waves take every 16th slice each, added in order.
struct SetupSum {
  const double* part;
  const double* kg;
  int ns;
  long n;
  double* mt;
  double* k0;
};
struct SetupSum2 {
  SetupSum s[2];
};
__global__ __launch_bounds__(1024) void setup_sum_kernel(SetupSum2 sets, int G) {
  __shared__ double red[16][64];
  const SetupSum& p = sets.s[blockIdx.y];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool last = blockIdx.x == gridDim.x - 1;
  const long e = blockIdx.x * 64L + lane;
  double s = 0.0;
  if (last) {
    for (int g = threadIdx.x; g < G; g += 1024) s += p.kg[g];
    s = wave_sum(s);
  } else if (e < p.n) {
#pragma unroll 4
    for (int i = wave; i < p.ns; i += 16) s += p.part[i * p.n + e];
  }
  red[wave][lane] = s;
  __syncthreads();
  if (wave > 0) return;
  double t = 0.0;
#pragma unroll
  for (int i = 0; i < 16; ++i) t += red[i][lane];
  if (last) {
    if (lane == 0) *p.k0 = t;
  } else if (e < p.n) {
    p.mt[e] = t;
  }
}

// The set-up of a few occupied orbitals, one work-group a Cholesky index g: f0 and
// rot_chol_g Q in LDS, then c0, tr(f0 f0), this g's part of M and its rows of the
// packed A (zero in the tile rows past the chunk's last g).  Thread (c, i0) forms
// column c of rows i0, i0 + ni, ...  Bound: launches, of which the general products
// take seven a spin.  Intermediates and job of a run (UHF N = 20, O = 6 / 5, G = 80,
// 100 walkers): 1.27 ms before, 0.96 now; RHF N = 10, O = 5, G = 27, which needs no
// factors at all: 0.76 and 0.55.
constexpr int kSetupMaxN = 128, kSetupMaxO = 24;
struct SetupSmall {
  const double *rc, *Q, *P;
  int O, gw, RB, n8;
  double *c0, *kg, *part;
  double2* a;
};
struct SetupSmall2 {
  SetupSmall s[2];
};
__global__ __launch_bounds__(256) void setup_small_kernel(SetupSmall2 sets, int N, int G) {
  extern __shared__ double sh[];
  __shared__ double red[8];
  const SetupSmall& p = sets.s[blockIdx.y];
  const int O = p.O, Nv = N - O, tid = threadIdx.x, g = blockIdx.x;
  double* rc = sh;           // (O, N)
  double* rv = rc + O * N;   // (O, Nv)
  double* f = rv + O * Nv;   // (O, O)
  for (int e = tid; e < O * N; e += 256) rc[e] = p.rc[(long)g * O * N + e];
  __syncthreads();
  const int ni = 256 / N, i0 = tid / N, c = tid - i0 * N;  // ni >= 2
  if (i0 < ni) {
    const double* b = c < O ? p.P + c : p.Q + (c - O);
    const int ld = c < O ? O : Nv;
    double acc[kSetupMaxO / 2];
#pragma unroll
    for (int k = 0; k < kSetupMaxO / 2; ++k) acc[k] = 0.0;
#pragma unroll 8
    for (int r = 0; r < N; ++r) {
      const double x = b[(long)r * ld];
#pragma unroll
      for (int k = 0; k < kSetupMaxO / 2; ++k)
        if (i0 + k * ni < O) acc[k] += rc[(i0 + k * ni) * N + r] * x;
    }
#pragma unroll
    for (int k = 0; k < kSetupMaxO / 2; ++k) {
      const int i = i0 + k * ni;
      if (i >= O) continue;
      if (c < O)
        f[i * O + c] = acc[k];
      else
        rv[i * Nv + c - O] = acc[k];
    }
  }
  __syncthreads();
  double t = 0.0, kk = 0.0;
  for (int e = tid; e < O * O; e += 256) {
    const int i = e / O, j = e - i * O;
    kk += f[e] * f[j * O + i];
    if (i == j) t += f[e];
  }
  t = wave_sum(t);
  kk = wave_sum(kk);
  if ((tid & 63) == 0) {
    red[tid >> 6] = t;
    red[4 + (tid >> 6)] = kk;
  }
  __syncthreads();
  if (tid == 0) {
    p.c0[g] = red[0] + red[1] + red[2] + red[3];
    p.kg[g] = red[4] + red[5] + red[6] + red[7];
  }
  for (int e = tid; e < O * Nv; e += 256) {
    const int i = e / Nv, v = e - i * Nv;
    double m = 0.0;
    for (int k = 0; k < O; ++k) m += f[i * O + k] * rv[k * Nv + v];
    p.part[(long)g * O * Nv + e] = m;
  }
  const int ck = g / p.gw, row0 = (g - ck * p.gw) * O;
  const bool fill = g == G - 1 || g == ck * p.gw + p.gw - 1;
  const int rows = fill ? 16 * p.RB - row0 : O, nk = 4 * p.n8;
  double2* out = p.a + (long)ck * p.RB * p.n8 * 64;
  for (int e = tid; e < rows * nk; e += 256) {
    const int i = e / nk, sq = e - i * nk, k = 2 * sq, row = row0 + i;
    double2 v = {0.0, 0.0};
    if (i < O) {
      if (k < Nv) v.x = rv[i * Nv + k];
      if (k + 1 < Nv) v.y = rv[i * Nv + k + 1];
    }
    out[((row >> 4) * p.n8 + (sq >> 2)) * 64 + (sq & 3) * 16 + (row & 15)] = v;
  }
}

unsigned blocks(long n) { return (unsigned)((n + 255) / 256); }

int mm(hipStream_t st, int M, int N, int K, const double* A, long lda, bool at, const double* B, long ldb, double* C,
       long ldc, double alpha, double beta, double* ws, long ws_elems) {
  Gemm g;
  g.M = M;
  g.N = N;
  g.K = K;
  g.A = A;
  g.lda = lda;
  g.a_trans = at;
  g.B = B;
  g.ldb = ldb;
  g.C = C;
  g.ldc = ldc;
  g.alpha = double2{alpha, 0.0};
  g.beta = double2{beta, 0.0};
  g.ws = ws;
  g.ws_elems = ws_elems;
  return gemm_f64(g, st);
}

template <int MB, int NB, int WR, int WC>
int launch(const ExF64& p, long grid, hipStream_t st) {
  constexpr size_t stage = sizeof(double2) * 2 * kPairs * 16 * NB * WC;
  const size_t bytes = std::max(stage, sizeof(double) * p.lds_elems);
  static std::atomic<uint64_t> raised{0};
  AFQ_TRY(raise_lds(reinterpret_cast<const void*>(exchange_f64_kernel<MB, NB, WR, WC>),
                    std::max(stage, tile_room(MB, NB, WR * WC)), raised, "exchange"));
  hipLaunchKernelGGL((exchange_f64_kernel<MB, NB, WR, WC>), dim3((unsigned)grid), dim3(64 * WR * WC), bytes, st, p);
  return launch_status("exchange_f64_kernel");
}

}  // namespace

// Few walkers: up to what theta_kernel reads of Q, each walker anew.  An energy with
// a product, a packing and a sum for theta, and with theta_kernel, at G = 400:
// N = 80, O = 20, 1 walker (0.2 MB) 75 and 58 us; N = 100, O = 20, 64 (20 MB) 187
// and 164, 512 (164 MB) 952 and 951; N = 200, O = 40, 128 (328 MB) 1233 and 1229,
// 256 (655 MB) 2344 and 2371.
constexpr double kFewBytes = 250.0e6;

// The tile: gw g's in 16 MB WR rows and wn walkers in 16 NB WC columns, chosen
// for the least padding.  One wave column up to O = 64 (all 2 O columns of a
// walker in one wave's 8 blocks); above, a whole f block takes eight waves.
// Sweep at O = 40 (ms a measurement of the N = 200 system above): 2 x 5 blocks
// on four waves with three work-groups a CU 12.2, with two 13.0; 3 x 5 on eight
// waves 12.3; 1 x 5 on eight 12.8; 3 x 5 on four 13.6.  At O = 60: 2 x 8 on four
// waves 67.2, 1 x 8 on eight 66.7, 2 x 8 on eight 68.5, 1 x 8 on four 74.0.
// O = 49 to 51: five g's in the 256 rows of eight waves (N = 250, G = 600, 128
// walkers 3.27 ms at O = 51, 3.95 with two in 128 rows).
// Share of the tile that is not padding: O <= 25 0.84 or more; 26 0.75, rising to 1
// at 32; 33 0.71, 38 0.94, 40 0.94, 43 0.80, 48 1; 49 0.84, 52 0.75, 57 0.79, 64 1;
// above, where a tile holds one f block, 65 0.46, 82 0.73, 96 1, 97 0.57, 112 0.77,
// 128 1.
ExF64Tile exchange_f64_tile(int O) {
  ExF64Tile best{};
  double top = -1.0;
  auto consider = [&](int MB, int NB, int WR, int WC) {
    const int rows = 16 * MB * WR, cols = 16 * NB * WC;
    const int gw = rows / O, wn = cols / (2 * O);
    if (gw < 1 || wn < 1) return;
    const double eff = (double)gw * O / rows * ((double)2 * O * wn / cols);
    if (eff > top * 1.02) {
      top = eff;
      best = ExF64Tile{MB, NB, WR, WC, gw, wn};
    }
  };
  if (O <= 64) {
    for (int nb = 8; nb >= 5; --nb) consider(2, nb, 4, 1);
    consider(3, 5, 4, 1);
    consider(3, 6, 4, 1);
    if (O > 48 && O <= 51) consider(2, 7, 8, 1);
  } else {
    consider(3, 3, 2, 4);
    consider(4, 4, 2, 4);
  }
  return best;
}

// Few walkers leave most of the tile's columns, or of the CUs, idle: then the
// widest of the narrower tiles that fills both, or else the narrowest (an energy at
// N = 60, O = 12, G = 144, 4 walkers 42 -> 35 us; N = 96, O = 16, G = 400, 4 walkers
// 62 -> 50).
ExF64Tile exchange_f64_tile(int O, int W, int G) {
  ExF64Tile t = exchange_f64_tile(O);
  const long nchunk = exchange_f64_nchunk(O, G);
  for (int nb = 4; nb >= 2; --nb) {
    const bool full = W >= t.wn && nchunk * ((W + t.wn - 1) / t.wn) >= 256;
    if (full || t.WC > 1 || 16 * nb < 2 * O) break;
    t.NB = nb;
    t.wn = 16 * nb / (2 * O);
  }
  return t;
}

long exchange_f64_most_few(int O, int N) {
  if (N <= O) return 0;
  const double bytes = 8.0 * N * (N - O) * ((O + kThetaRows - 1) / kThetaRows);
  return (long)std::min(65535.0, kFewBytes / bytes);
}
bool exchange_f64_few(int O, int N, int W) { return W <= exchange_f64_most_few(O, N); }
static int theta_blocks(int O, int N) { return (2 * exchange_f64_npairs(N - O) + 63) / 64; }
int exchange_f64_slots(int O, int N, int G) {
  return exchange_f64_nchunk(O, G) + std::max(1, (O + kThetaRows - 1) / kThetaRows * theta_blocks(O, N));
}

int exchange_f64_theta(const ExTheta* sets, int nsets, int N, int G, int W, double fac, double2* ene1,
                       hipStream_t st) {
  if (nsets < 1) return AFQ_OK;
  ThetaArgs a{};
  int rows = 0;
  for (int i = 0; i < nsets; ++i) {
    const ExTheta& x = sets[i];
    const ExF64Tile t = exchange_f64_tile(x.O, W, G);
    a.s[i] = ThetaSet{x.green, x.Q, x.mt, x.k0, x.rh1, x.O, theta_blocks(x.O, N), t.wn, 8 * t.NB * t.WC,
                      exchange_f64_npairs(N - x.O), exchange_f64_nchunk(x.O, G), exchange_f64_slots(x.O, N, G),
                      x.thetap, x.kpart};
    rows = std::max(rows, x.O);
  }
  a.nsets = nsets;
  a.N = N;
  a.fac = fac;
  a.ene1 = ene1;
  const dim3 grid(a.s[0].nx + a.s[1].nx + (ene1 ? 1 : 0), (rows + kThetaRows - 1) / kThetaRows, W);
  hipLaunchKernelGGL(theta_kernel, grid, dim3(64 * kThetaWaves), 0, st, a);
  return launch_status("theta_kernel");
}

int exchange_f64_nchunk(int O, int G) {
  const ExF64Tile t = exchange_f64_tile(O);
  return (G + t.gw - 1) / t.gw;
}

int exchange_f64_npairs(int Nv) { return ((Nv + 7) / 8 + kSteps - 1) / kSteps * kPairs; }

// For up to W walkers: the widest tile, and the narrower ones up to the walkers
// (256 work-groups of the widest, at most) that take them.
long exchange_f64_b_elems(int O, int N, int W) {
  ExF64Tile t = exchange_f64_tile(O);
  long n = exchange_thetap_elems(t, N - O, W);
  const int few = std::min(W, 256 * t.wn);
  for (t.NB = 4; t.WC == 1 && t.NB >= 2 && 16 * t.NB >= 2 * O; --t.NB) {
    t.wn = 16 * t.NB / (2 * O);
    n = std::max(n, exchange_thetap_elems(t, N - O, few));
  }
  return n;
}

long exchange_f64_a_elems(int O, int N, int G) {
  const ExF64Tile t = exchange_f64_tile(O);
  return (long)exchange_f64_nchunk(O, G) * t.MB * t.WR * ((N - O + 7) / 8) * 128;
}

// g's of one setup pass: a multiple of the tile's, about 64 MB of products.
// M is summed in slices of g's, so that its O x Nv product has work-groups
// enough.
struct Setup {
  int gc, gs, ns;
};
static Setup setup_pass(int O, int N, int G) {
  const ExF64Tile t = exchange_f64_tile(O);
  const long per = (long)O * (N + O) * (long)sizeof(double);
  const long n = std::max(1L, (64L << 20) / per / t.gw) * t.gw;
  Setup u;
  u.gc = (int)std::min(n, (long)exchange_f64_nchunk(O, G) * t.gw);
  const int first = std::min(u.gc, G);
  u.gs = std::max(1, first / 64);
  u.ns = first / u.gs;
  return u;
}

// Sizes of setup_small_kernel (48 KB of LDS at most).
static bool setup_small(int O, int N) { return N <= kSetupMaxN && O <= kSetupMaxO; }

static long trial_elems(int O, int N) { return 2L * O * N + O + (long)O * O; }

long exchange_f64_tmp_elems(int O, int N, int G) {
  const Setup u = setup_pass(O, N, G);
  const long chol = setup_small(O, N) ? 2L * G * O * (N - O)
                                      : (long)u.gc * O * (N - O) + 2L * u.gc * O * O + (long)u.ns * O * (N - O);
  return std::max(chol, 2 * trial_elems(O, N));
}

int exchange_f64_set_trial(const ExTrial* sets, int nsets, int N, double* tmp, hipStream_t st) {
  if (nsets < 1) return AFQ_OK;
  TrialQR2 q{};
  int omax = 0;
  for (int i = 0; i < nsets; ++i) {
    const int O = sets[i].O;
    double* V = tmp;
    double* tau = V + (long)O * N;
    double* RT = tau + O;
    double* Q1 = RT + (long)O * O;
    q.s[i] = TrialQR{sets[i].mo, O, V, tau, RT, Q1, sets[i].Q, sets[i].P};
    tmp += trial_elems(O, N);
    omax = std::max(omax, O);
  }
  const size_t bytes = sizeof(double) * N * omax;
  constexpr size_t most = 152 * 1024;
  if (bytes <= most) {
    static std::atomic<uint64_t> raised{0};
    AFQ_TRY(raise_lds(reinterpret_cast<const void*>(householder_kernel<true>), most, raised, "householder"));
    hipLaunchKernelGGL(householder_kernel<true>, dim3(1, nsets), dim3(1024), bytes, st, q, N);
  } else {
    hipLaunchKernelGGL(householder_kernel<false>, dim3(1, nsets), dim3(1024), 0, st, q, N);
  }
  AFQ_TRY(launch_status("householder_kernel"));
  const dim3 grid(N, nsets);
  if (N <= 64)
    hipLaunchKernelGGL(basis_kernel<1>, grid, dim3(64), 0, st, q, N);
  else if (N <= 128)
    hipLaunchKernelGGL(basis_kernel<2>, grid, dim3(64), 0, st, q, N);
  else if (N <= 512)
    hipLaunchKernelGGL(basis_kernel<8>, grid, dim3(64), 0, st, q, N);
  else
    hipLaunchKernelGGL(basis_kernel<0>, grid, dim3(64), 0, st, q, N);
  AFQ_TRY(launch_status("basis_kernel"));
  hipLaunchKernelGGL(dual_kernel, dim3(N, nsets), dim3(64), 0, st, q);
  return launch_status("dual_kernel");
}

// One spin by general products, passes of gc g's at a time; leaves ns slices of M
// in *part_out and tr(f0 f0) in kg.
static int set_chol_general(const ExChol& x, int N, int G, double* kg, double* tmp, double* ws, long ws_elems,
                            double** part_out, hipStream_t st) {
  const int O = x.O;
  const ExF64Tile t = exchange_f64_tile(O);
  const int Nv = N - O, n8 = (Nv + 7) / 8, RB = t.MB * t.WR;
  const Setup u = setup_pass(O, N, G);
  const int gc = u.gc;
  double* rcv = tmp;
  double* f0 = rcv + (long)gc * O * Nv;
  double* ft = f0 + (long)gc * O * O;
  double* part = ft + (long)gc * O * O;
  *part_out = part;
  for (int g0 = 0; g0 < G; g0 += gc) {
    const int gn = std::min(gc, G - g0);
    const double* r = x.rc + (long)g0 * O * N;
    AFQ_TRY(mm(st, gn * O, O, N, r, N, false, x.P, O, f0, O, 1.0, 0.0, nullptr, 0));
    hipLaunchKernelGGL(occ_terms_kernel, dim3(gn), dim3(256), 0, st, f0, O, x.c0 + g0, kg + g0, ft);
    AFQ_TRY(launch_status("occ_terms_kernel"));
    if (Nv == 0) continue;
    AFQ_TRY(mm(st, gn * O, Nv, N, r, N, false, x.Q, Nv, rcv, Nv, 1.0, 0.0, nullptr, 0));
    Gemm m;  // slice i of M: the g's [i gs, (i + 1) gs) of every pass
    m.M = O;
    m.N = Nv;
    m.K = u.gs * O;
    m.batch = std::min(gn / u.gs, u.ns);
    m.a_trans = true;
    m.A = ft;
    m.lda = O;
    m.sA = (long)u.gs * O * O;
    m.B = rcv;
    m.ldb = Nv;
    m.sB = (long)u.gs * O * Nv;
    m.C = part;
    m.ldc = Nv;
    m.sC = (long)O * Nv;
    m.beta = double2{g0 > 0 ? 1.0 : 0.0, 0.0};
    if (m.batch > 0) AFQ_TRY(gemm_f64(m, st));
    const int done = m.batch * u.gs;
    if (done < gn)
      AFQ_TRY(mm(st, O, Nv, (gn - done) * O, ft + (long)done * O * O, O, true, rcv + (long)done * O * Nv, Nv, part, Nv,
                 1.0, 1.0, ws, ws_elems));
    const long nck = (gn + t.gw - 1) / t.gw;
    const long n = nck * RB * n8 * 64;
    hipLaunchKernelGGL(pack_a_kernel, dim3(blocks(n)), dim3(256), 0, st, rcv, O, Nv, t.gw, gn, RB, n8, nck,
                       reinterpret_cast<double2*>(x.a + (long)(g0 / t.gw) * RB * n8 * 128));
    AFQ_TRY(launch_status("pack_a_kernel"));
  }
  return AFQ_OK;
}

static int set_sums(const SetupSum2& q, int nsets, int G, hipStream_t st) {
  const long n = std::max(q.s[0].n, q.s[1].n);
  hipLaunchKernelGGL(setup_sum_kernel, dim3((unsigned)((n + 63) / 64 + 1), nsets), dim3(1024), 0, st, q, G);
  return launch_status("setup_sum_kernel");
}

int exchange_f64_set_chol(const ExChol* sets, int nsets, int N, int G, double* kg, double* tmp, double* ws,
                          long ws_elems, hipStream_t st) {
  SetupSmall2 p{};
  SetupSum2 q{};
  int ns = 0;
  double* part = tmp;
  size_t lds = 0;
  for (int i = 0; i < nsets; ++i) {
    const ExChol& x = sets[i];
    if (!setup_small(x.O, N)) continue;
    const ExF64Tile t = exchange_f64_tile(x.O);
    const long n = (long)x.O * (N - x.O);
    double* k = kg + ns * (long)G;
    p.s[ns] = SetupSmall{x.rc, x.Q, x.P, x.O, t.gw, t.MB * t.WR, (N - x.O + 7) / 8, x.c0, k, part,
                         reinterpret_cast<double2*>(x.a)};
    q.s[ns++] = SetupSum{part, k, G, n, x.mt, x.k0};
    part += G * n;
    lds = std::max(lds, sizeof(double) * (2 * (size_t)x.O * N));
  }
  if (ns > 0) {
    hipLaunchKernelGGL(setup_small_kernel, dim3(G, ns), dim3(256), lds, st, p, N, G);
    AFQ_TRY(launch_status("setup_small_kernel"));
    AFQ_TRY(set_sums(q, ns, G, st));
  }
  for (int i = 0; i < nsets; ++i) {
    const ExChol& x = sets[i];
    if (setup_small(x.O, N)) continue;
    AFQ_TRY(set_chol_general(x, N, G, kg, tmp, ws, ws_elems, &part, st));
    SetupSum2 one{};
    one.s[0] = SetupSum{part, kg, setup_pass(x.O, N, G).ns, (long)x.O * (N - x.O), x.mt, x.k0};
    AFQ_TRY(set_sums(one, 1, G, st));
  }
  return AFQ_OK;
}

int k_exchange_f64(const double* a, const double* Q, const double* c0, const double* mt, const double* k0,
                   const double2* green, double2* theta, double2* thetap, int O, int N, int G, int W, double2* coul,
                   double2* kpart, int* nch_out, hipStream_t st) {
  if (O < 1 || O > kExchangeF64MaxO) return fail(AFQ_E_UNSUPPORTED, "exchange kernel supports 1 <= nocc <= 128");
  const ExF64Tile t = exchange_f64_tile(O, W, G);
  ExF64 p;
  p.a = a;
  p.theta = thetap;
  p.c0 = c0;
  p.O = O;
  p.Nv = N - O;
  p.n8 = (p.Nv + 7) / 8;
  p.G = G;
  p.W = W;
  p.gw = t.gw;
  p.wn = t.wn;
  p.nwg = (W + t.wn - 1) / t.wn;
  p.nchunk = exchange_f64_nchunk(O, G);
  p.coul = coul;
  p.kpart = kpart;
  const long ld = 16L * t.NB * t.WC + 2;
  const long room = (long)(tile_room(t.MB, t.NB, t.WR * t.WC) / sizeof(double));
  p.gp = (int)std::min((long)t.gw, room / (O * ld));
  p.strip = O;
  if (p.gp == 0) {  // one g in strips: strip rows, and the strip's columns of all rows
    p.gp = 1;
    p.strip = (int)((room - 2 * O) / (ld + 2 * O));
  }
  p.lds_elems = p.strip < O ? p.strip * ld + O * (2L * p.strip + 2) : p.gp * O * ld;
  const int nslab = (p.n8 + kSteps - 1) / kSteps;
  p.kstride = exchange_f64_few(O, N, W) ? exchange_f64_slots(O, N, G) : p.nchunk + 1;
  *nch_out = p.kstride;
  if (green && p.Nv > 0) {
    // theta^T: the rows (w, j) of all walkers' G times Q
    Gemm g;
    g.M = W * O;
    g.N = p.Nv;
    g.K = N;
    g.a_cplx = true;
    g.A = green;
    g.lda = N;
    g.B = Q;
    g.ldb = p.Nv;
    g.C = theta;
    g.ldc = p.Nv;
    AFQ_TRY(gemm_f64(g, st));
    const long n = (long)p.nwg * nslab * kPairs * 8 * t.NB * t.WC;
    hipLaunchKernelGGL(pack_b_kernel, dim3(blocks(n)), dim3(256), 0, st, theta, O, p.Nv, t.wn, W, 8 * t.NB * t.WC,
                       nslab, n, thetap);
    AFQ_TRY(launch_status("pack_b_kernel"));
  }
  // chunks per group: a slice of A that stays in one XCD's L2 beside theta
  const long chunk_bytes = 16L * t.MB * t.WR * 8 * p.n8 * (long)sizeof(double);
  p.cpg = (int)std::max(1L, std::min((long)p.nchunk, (2560L * 1024) / std::max(1L, chunk_bytes)));
  const long ngroups = (p.nchunk + p.cpg - 1) / p.cpg;
  p.T8 = (ngroups * p.cpg * (long)p.nwg + 7) / 8;
  const long grid = 8 * p.T8;
  if (grid > 0x7fffffffL) return fail(AFQ_E_UNSUPPORTED, "exchange grid too large");
  if (green) {
    hipLaunchKernelGGL(exchange_occ_kernel, dim3(W), dim3(256), 0, st, theta, mt, k0, (long)p.Nv * O, p.nchunk, kpart);
    AFQ_TRY(launch_status("exchange_occ_kernel"));
  }
#define EXF64(mb, nb, wr, wc) \
  if (t.MB == mb && t.NB == nb && t.WR == wr && t.WC == wc) return launch<mb, nb, wr, wc>(p, grid, st)
  EXF64(2, 8, 4, 1);
  EXF64(2, 7, 4, 1);
  EXF64(2, 6, 4, 1);
  EXF64(2, 5, 4, 1);
  EXF64(2, 4, 4, 1);
  EXF64(2, 3, 4, 1);
  EXF64(2, 2, 4, 1);
  EXF64(3, 2, 4, 1);
  EXF64(3, 3, 4, 1);
  EXF64(3, 4, 4, 1);
  EXF64(3, 5, 4, 1);
  EXF64(3, 6, 4, 1);
  EXF64(2, 7, 8, 1);
  EXF64(3, 3, 2, 4);
  EXF64(4, 4, 2, 4);
#undef EXF64
  return fail(AFQ_E_UNSUPPORTED, "exchange: no tile for this nocc");
}

}  // namespace afq

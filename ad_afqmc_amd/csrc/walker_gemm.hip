// FP64 products of a step that run over all walkers at once: the force bias and
// the VHS (ad_afqmc/wavefunctions.py:202-262, ad_afqmc/propagation.py:196-203).
//
// Both multiply a real matrix that all walkers share (rot_chol: rows of K
// contiguous elements; packed L: K rows) by the walkers' complex vectors, so
// the shared matrix gives the rows of a real product and (walker, re/im) the
// columns: one MFMA a block and 4-deep step, no multiplication by zero parts.
// A work-group of WR x WC waves of MB x NB blocks stages 16-deep slabs of both
// operands in two LDS buffers, the next slab in registers while the current one
// is multiplied.  LDS rows are swizzled in 16-byte units (unit ^ row % 8), so
// fragment reads down a column of rows are free of bank conflicts.
//
// Waves of 64 x 32 walkers (four to a work-group, two work-groups a CU) where
// there are more than 32 walkers: at MB NB = 8 and four waves a SIMD the
// prefetched slab does not fit the 128 registers and the loads sink behind the
// product.  Whole slabs are fetched by pointers that only move; clamping to the
// end of K is left to the last one (it had cost 6% as vector work in every slab).
//
// The force bias has few output tiles and a long K (all occupied x orbital
// pairs of both spins): K is cut into slices, each slice's partial sums go to a
// workspace and a second kernel adds them in order.
//
// Bound: the FP64 matrix cores (57-58 of the 72.8 TF/s that an 8192^3 product
// reaches; the clock falls to 2.2 GHz under this load); for few walkers the
// reads of rot_chol and L.  Measured, before (the general product kernel, split
// over K, and strided 16-byte stores of a packed triangle) and now:
//   force bias  N=200 O=40 G=1200 W=512: 567 -> 400 us; N=300 O=60+58 G=2000
//               W=256: 1865 -> 1270; N=100 O=20 G=500 W=256: 255 -> 42;
//   VHS         N=200: 1110 -> 1054 us; N=300: 1806 -> 1697; N=100: 152 -> 79,
// and the propagator reads the VHS by blocks in its own order, which took it
// from 820 to 786, 2578 to 2430 and 143 to 101 us.
#include "walker_gemm.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace afq {
namespace {

constexpr int KS = 16;

typedef double v2d __attribute__((ext_vector_type(2)));
typedef v2d v2du __attribute__((aligned(8)));

struct WgArgs {
  const double* A[2];
  const double2* X[2];
  long lda[2], ldx[2], K[2];  // K per part (the spins of the force bias)
  int M, W;                   // rows of the product, walkers
  int nz0, nz;                // slices of part 0 and of both: those from nz0 on belong to part 1
  long kc[2];                 // depth of a slice, per part
  int tm, tn;
  long T8;
  double* out;
  double scale;
  int R;                      // VHS epilogue
};

// AK: A row m holds its K elements contiguously (lda = row stride); else A row
// k holds the M elements.  VHS: epilogue into the propagator's blocks.
template <bool AK, int MB, int NB, int WR, int WC, bool VHS>
__global__ __launch_bounds__(64 * WR * WC, MB * NB <= 8 ? 4 : 2) void walker_gemm_kernel(WgArgs p) {
  constexpr int NT = 64 * WR * WC, BM = 16 * MB * WR, BW = 8 * NB * WC;
  constexpr int UA = BM * 8 / NT, UB = (BW * KS + NT - 1) / NT;
  static_assert(UA * NT == BM * 8, "A slab must split evenly");
  __shared__ v2d As[2][BM * 8];
  __shared__ v2d Bs[2][BW * KS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave / WC, wc = wave % WC, q = lane >> 4, c16 = lane & 15;
  const long L = (long)(blockIdx.x & 7) * p.T8 + (blockIdx.x >> 3);
  const long tiles = (long)p.tm * p.tn;
  const int z = (int)(L / tiles);
  const int t = (int)(L - (long)z * tiles);
  if (z >= p.nz) return;  // uniform
  const int part = z >= p.nz0;
  const long kc = p.kc[part], K = p.K[part];
  const long k0 = (long)(z - (part ? p.nz0 : 0)) * kc, k1 = min(K, k0 + kc);
  const int m0 = (t / p.tn) * BM, w0 = (t % p.tn) * BW;
  const double* A = p.A[part];
  const double2* X = p.X[part];
  const long lda = p.lda[part], ldx = p.ldx[part];

  // This thread's 16-byte units of a slab (rows past M and walkers past W
  // repeat the last: their results are dropped), as pointers that move with the
  // slabs.  kr is what remains of the slice from a slab on: past it A is zero
  // and the loads stay on its last element.
  const double* pa[UA];
  const v2d* pb[UB];
#pragma unroll
  for (int u = 0; u < UA; ++u) {
    const int e = tid + u * NT;
    pa[u] = AK ? A + min(m0 + (e >> 3), p.M - 1) * lda + k0 + 2 * (e & 7)
               : A + (k0 + e / (BM / 2)) * lda + m0 + 2 * (e % (BM / 2));
  }
#pragma unroll
  for (int u = 0; u < UB; ++u) {
    const int e = tid + u * NT;
    pb[u] = reinterpret_cast<const v2d*>(X) + min(w0 + (e >> 4), p.W - 1) * ldx + k0 + (e & 15);
  }
  v2d ra[UA], rb[UB];
  auto fetch = [&](int kr, auto full) {
#pragma unroll
    for (int u = 0; u < UA; ++u) {
      const int e = tid + u * NT, kk = AK ? 2 * (e & 7) : e / (BM / 2);
      const int back = full ? 0 : min(kr - 1 - kk, 0);
      if (AK) {
        if (full) ra[u] = *reinterpret_cast<const v2du*>(pa[u]);
        else ra[u] = v2d{pa[u][back], pa[u][min(kr - 1 - kk, 1)]};
        pa[u] += KS;
      } else {
        ra[u] = *reinterpret_cast<const v2d*>(pa[u] + back * lda);
        pa[u] += KS * lda;
      }
    }
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      rb[u] = pb[u][full ? 0 : min(kr - 1 - ((tid + u * NT) & 15), 0)];
      pb[u] += KS;
    }
  };
  auto stash = [&](int kr, int buf, auto full) {
#pragma unroll
    for (int u = 0; u < UA; ++u) {
      const int e = tid + u * NT, kk = AK ? 2 * (e & 7) : e / (BM / 2);
      v2d v = ra[u];
      if (!full && kk >= kr) v = v2d{0.0, 0.0};
      if (!full && AK && kk + 1 >= kr) v.y = 0.0;
      As[buf][AK ? (e >> 3) * 8 + ((e & 7) ^ ((e >> 3) & 7)) : e] = v;
    }
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      const int e = tid + u * NT, w = e >> 4;
      if (UB * NT == BW * KS || w < BW) Bs[buf][w * KS + ((e & 15) ^ (w & 7))] = rb[u];
    }
  };

  v4d acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  auto multiply = [&](int buf) {
    const v2d* a = As[buf];
    const double* b = reinterpret_cast<const double*>(Bs[buf]);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      v2d av[MB], bv[NB];  // k = 8 h + 2 q and the next
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const int r = (wr * MB + i) * 16 + c16;
        if (AK) {
          av[i] = a[r * 8 + ((4 * h + q) ^ (r & 7))];
        } else {
          const double* s = reinterpret_cast<const double*>(a) + (8 * h + 2 * q) * BM + r;
          av[i] = v2d{s[0], s[BM]};
        }
      }
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int w = (wc * NB + j) * 8 + (c16 >> 1), kk = 8 * h + 2 * q;
        bv[j].x = b[2 * (w * KS + (kk ^ (w & 7))) + (c16 & 1)];
        bv[j].y = b[2 * (w * KS + ((kk + 1) ^ (w & 7))) + (c16 & 1)];
      }
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i].x, bv[j].x, acc[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i].y, bv[j].y, acc[i][j], 0, 0, 0);
    }
  };
  const int depth = (int)(k1 - k0);
  const std::true_type full{};
  const std::false_type last{};
  fetch(depth, last);
  stash(depth, 0, last);
  __syncthreads();
  int buf = 0, k = KS;
  for (; k + KS <= depth; k += KS) {
    fetch(KS, full);
    __builtin_amdgcn_sched_barrier(0);  // or the loads sink to where they are stored
    multiply(buf);
    buf ^= 1;
    stash(KS, buf, full);
    __syncthreads();
  }
  if (k < depth) {
    fetch(depth - k, last);
    __builtin_amdgcn_sched_barrier(0);
    multiply(buf);
    buf ^= 1;
    stash(depth - k, buf, last);
    __syncthreads();
  }
  multiply(buf);

  // element v of block (i, j): row m0 + 16 (wr MB + i) + q + 4 v, column (walker, re/im)
  const int pt = c16 & 1;
  if constexpr (VHS) {
    // Times i sqrt(dt): the real part of x.L is the imaginary part of the VHS.
    // The tile's rows are rows r0.. of one 16 x 16 block (ib, jb); 8 WC walkers
    // at a time pass through LDS, so that the block and its mirror both go out
    // in runs of 128 and 256 bytes (straight from the lanes they are 16-byte
    // pieces, and a step is 1.2% slower at N=200).  Units swizzled by walker and row.
    static_assert(WC == 2, "the first slab buffers hold 16 walkers of the tile");
    constexpr int RB = BM / 16;
    v2d* stage = As[0];
    const double sc = pt ? -p.scale : p.scale;
    const int r0 = (m0 >> 4) & 15;
    int ib, jb;
    sym_block(m0 >> 8, &ib, &jb);
    const long bl = 256L * (ib * p.R + jb), bm = 256L * (jb * p.R + ib), per = 256L * p.R * p.R;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      __syncthreads();
      const int wl = wc * 8 + (c16 >> 1);
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int r = wr * MB + i;
          reinterpret_cast<double*>(stage + wl * BM + r * 16 + ((q + 4 * v) ^ ((wl ^ r) & 7)))[1 - pt] = sc * acc[i][j][v];
        }
      __syncthreads();
#pragma unroll
      for (int e = tid; e < 16 * BM; e += NT) {
        const int r = e % RB, c = e / RB & 15, x = e / BM, w = w0 + ((x >> 3) * NB + j) * 8 + (x & 7);
        if (w < p.W)
          reinterpret_cast<v2d*>(p.out)[w * per + bl + (c & 3) * 64 + (c >> 2) * 16 + r0 + r] =
              stage[x * BM + r * 16 + (c ^ ((x ^ r) & 7))];
      }
      if (ib != jb) {
#pragma unroll
        for (int e = tid; e < 16 * BM; e += NT) {
          const int c = e & 15, r = e / 16 % RB, x = e / BM, w = w0 + ((x >> 3) * NB + j) * 8 + (x & 7);
          if (w < p.W)
            reinterpret_cast<v2d*>(p.out)[w * per + bm + ((r0 + r) & 3) * 64 + ((r0 + r) >> 2) * 16 + c] =
                stage[x * BM + r * 16 + (c ^ ((x ^ r) & 7))];
        }
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int w = w0 + (wc * NB + j) * 8 + (c16 >> 1);
      if (w >= p.W) continue;
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int m = m0 + (wr * MB + i) * 16 + q + 4 * v;
          if (m < p.M) p.out[((long)z * p.W + w) * 2 * p.M + 2 * m + pt] = acc[i][j][v];
        }
    }
  }
}

// out = fac sum_z ws[z]
__global__ void slices_kernel(const double2* __restrict__ ws, int nz, long n, double fac, double2* __restrict__ out) {
  const long e = blockIdx.x * 256L + threadIdx.x;
  if (e >= n) return;
  double2 s = {0.0, 0.0};
#pragma unroll 4
  for (int z = 0; z < nz; ++z) {
    const double2 v = ws[z * n + e];
    s.x += v.x;
    s.y += v.y;
  }
  out[e] = double2{fac * s.x, fac * s.y};
}

// Walkers of a tile: the least of 16, 32 and 64 that holds them all, since
// what a tile has beyond W is multiplied for nothing.
int walkers_of(int W) { return W > 32 ? 64 : W > 16 ? 32 : 16; }

struct Slices {
  long kc[2];
  int nz[2];
};
// Slices of the force bias, in both parts about equally deep: the least time of
// the rounds of 512 work-groups (two a CU), in MFMA slabs of 3.8 us for a 128 x
// 128 tile when two share a CU, plus writing and reading the partial sums.
Slices fb_slices(int W, int G, long K0, long K1, long ws_elems) {
  const int bw = walkers_of(W);
  const double tiles = (double)((G + 127) / 128) * ((W + bw - 1) / bw);
  const double slab = 3.8 * bw / 64, part = 2.0 * 16.0 * W * G / 4.0e6;
  Slices best{};
  double top = 0.0;
  for (int n = 1; n <= 64; ++n) {
    Slices s{};
    const long K[2] = {K0, K1};
    s.nz[0] = K1 == 0 ? n : (int)std::min<long>(std::max<long>(1, std::lround((double)n * K0 / (K0 + K1))), std::max(1, n - 1));
    s.nz[1] = K1 == 0 ? 0 : std::max(1, n - s.nz[0]);
    for (int i = 0; i < 2 && K[i] > 0; ++i) {
      s.kc[i] = ((K[i] + s.nz[i] - 1) / s.nz[i] + KS - 1) / KS * KS;
      s.nz[i] = (int)((K[i] + s.kc[i] - 1) / s.kc[i]);
    }
    const int nz = s.nz[0] + s.nz[1];
    if (top > 0.0 && (long)nz * 2 * W * G > ws_elems) continue;
    const double t = std::ceil(tiles * nz / 512.0) * (std::max(s.kc[0], s.kc[1]) / KS * slab + 3.0) + nz * part;
    if (top == 0.0 || t < top) {
      best = s;
      top = t;
    }
  }
  return best;
}

template <bool AK, int MB, int NB, int WR, int WC, bool VHS>
int launch(WgArgs p, hipStream_t st) {
  constexpr int BM = 16 * MB * WR, BW = 8 * NB * WC;
  p.tm = (p.M + BM - 1) / BM;
  p.tn = (p.W + BW - 1) / BW;
  p.T8 = ((long)p.tm * p.tn * p.nz + 7) / 8;
  const long grid = 8 * p.T8;
  if (grid > 0x7fffffffL) return fail(AFQ_E_UNSUPPORTED, "walker product: grid too large");
  hipLaunchKernelGGL((walker_gemm_kernel<AK, MB, NB, WR, WC, VHS>), dim3((unsigned)grid), dim3(64 * WR * WC), 0, st, p);
  return launch_status("walker_gemm_kernel");
}

}  // namespace

long force_bias_f64_ws(int W, int G, long K0, long K1) {
  const Slices s = fb_slices(W, G, K0, K1, 1L << 40);
  return (long)(s.nz[0] + s.nz[1]) * 2 * W * G;
}

int force_bias_f64(const ForceBias64& f, hipStream_t st) {
  const Slices s = fb_slices(f.W, f.G, f.K[0], f.nspin > 1 ? f.K[1] : 0, f.ws_elems);
  const int nz = s.nz[0] + s.nz[1];
  if ((long)nz * 2 * f.W * f.G > f.ws_elems) return fail(AFQ_E_INVALID, "force bias: workspace too small");
  WgArgs p{};
  for (int i = 0; i < f.nspin; ++i) {
    p.A[i] = f.rc[i];
    p.lda[i] = f.K[i];
    p.X[i] = f.green[i];
    p.ldx[i] = f.K[i];
    p.K[i] = f.K[i];
  }
  p.M = f.G;
  p.W = f.W;
  p.nz0 = s.nz[0];
  p.nz = nz;
  p.kc[0] = s.kc[0];
  p.kc[1] = s.kc[1];
  p.out = f.ws;
  switch (walkers_of(f.W)) {
    case 64: AFQ_TRY((launch<true, 4, 4, 2, 2, false>(p, st))); break;
    case 32: AFQ_TRY((launch<true, 2, 2, 4, 2, false>(p, st))); break;
    default: AFQ_TRY((launch<true, 2, 1, 4, 2, false>(p, st))); break;
  }
  const long n = (long)f.W * f.G;
  hipLaunchKernelGGL(slices_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                     reinterpret_cast<const double2*>(f.ws), nz, n, f.fac, f.out);
  return launch_status("slices_kernel");
}

long vhs_f64_elems(int N) {
  const long R = (N + 15) / 16;
  return 256 * R * R;
}

int vhs_f64(const double2* xs, const double* lp, int N, int G, int W, double sqdt, double2* out, hipStream_t st) {
  WgArgs p{};
  p.R = (N + 15) / 16;
  p.M = p.R * (p.R + 1) / 2 * 256;
  p.A[0] = lp;
  p.lda[0] = p.M;
  p.X[0] = xs;
  p.ldx[0] = G;
  p.K[0] = G;
  p.W = W;
  p.nz0 = p.nz = 1;
  p.kc[0] = G;
  p.out = reinterpret_cast<double*>(out);
  p.scale = sqdt;
  // Half-height tiles where the full ones leave CUs without their two
  // work-groups.  Half against full: N=120 W=30, 72 full tiles, 29 / 46 us;
  // N=150 W=64, 110, 50 / 86; N=100 W=256, 224, 79 / 86; N=220 W=128, 420, 287 / 275.
  const int bw = walkers_of(W);
  const long tiles = (long)(p.M / 128) * ((W + bw - 1) / bw);
  const bool half = tiles < 320;
  switch (bw) {
    case 64: return half ? launch<false, 1, 4, 4, 2, true>(p, st) : launch<false, 4, 4, 2, 2, true>(p, st);
    case 32: return half ? launch<false, 1, 2, 4, 2, true>(p, st) : launch<false, 2, 2, 4, 2, true>(p, st);
    default: return half ? launch<false, 1, 1, 4, 2, true>(p, st) : launch<false, 2, 1, 4, 2, true>(p, st);
  }
}

}  // namespace afq

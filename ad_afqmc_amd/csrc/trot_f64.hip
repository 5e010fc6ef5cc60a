// Fused FP64 propagator of a step with symmetric Cholesky vectors:
//   W <- E T_K(VHS) E W,   E = exp(-dt/2 h1),  T_K(V) = sum_n V^n / n!
// (ad_afqmc/propagation.py:154-176), one work-group for the whole chain of a
// slab of a walker's columns.  T_K is evaluated as t0 + V (t0 + V/2 (t0 + ...)),
// t0 = E W, so a product's accumulators are the only large register state: t0
// waits in memory and is added at the end of each product.
//
// A work-group of eight waves holds 16 NB real columns (8 NB complex ones, re
// and im interleaved) of the panel in LDS and multiplies by whole row blocks.
// With A = VHS complex, D[:, (j, re/im)] += Re A . B + Im A . B', B' the columns
// of B swapped in pairs with a sign, so a 16 x 16 block takes two MFMAs per
// 4-deep step and no column is padded but the last.  A's fragments go straight
// from memory to registers, 1 KB of consecutive bytes each, eight k ahead of
// their use; k = 4 q + t within a 16-deep block for lane group q and MFMA t, on
// both operands.
//
// Row blocks: every wave takes R / 8 of them, four more go to the first waves of
// the four SIMDs, and the last one to three are split by columns over the waves,
// so the SIMDs differ by one block at most (N = 200: 17 of 16.25 blocks, where
// whole row blocks would leave 20).
//
// Bound: the FP64 matrix cores, 8 N^2 c flops a term, and at N = 100 the reads of
// the VHS, once a term and slab (fetching two to four steps ahead instead of one
// was slower there, 143 -> 177 us).  Measured
// against one launch a product with the running sum in memory, per step: N = 200,
// 40 columns, 512 walkers 1.30 -> 0.82 ms (48 TFLOP/s); N = 300, 60 + 58 columns,
// 256 walkers 3.25 -> 2.58 ms; N = 100, 20 columns, 256 walkers 181 -> 143 us.
// With the VHS read in the order of the fragments: 0.79 and 2.43 ms, 87 us.
#include "trot_f64.h"

#include <cmath>
#include <type_traits>

namespace afq {
namespace {

constexpr int NT = 512, NWAVE = 8;
constexpr long kLdsMax = 156 * 1024;

struct TrotArgs {
  TrotF64 f;
  int R, nslab[2];
};

__device__ __forceinline__ double swap_pair(double x) {
  const long long v = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_mov_dpp((int)(v & 0xffffffffLL), 0xB1, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(v >> 32), 0xB1, 0xF, 0xF, true);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

template <int MB, int NB, int XB>
__global__ __launch_bounds__(NT, 2) void trot_f64_kernel(TrotArgs a) {
  constexpr int LDP = 16 * NB;
  extern __shared__ double P[];  // [16 R][LDP]
  const TrotF64& f = a.f;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane >> 4, c16 = lane & 15;
  const int N = f.N, R = a.R;
  // XCD x takes the walkers x, x + 8, ..., all slabs of one in a row
  const int S = a.nslab[0] + a.nslab[1];
  const long idx = blockIdx.x >> 3;
  const long w = (idx / S) * 8 + (blockIdx.x & 7);
  if (w >= f.W) return;  // uniform
  int slab = (int)(idx % S);
  const int s = slab >= a.nslab[0];
  slab -= s ? a.nslab[0] : 0;
  const int cs = f.c[s], ct = f.c[0] + (f.nspin > 1 ? f.c[1] : 0);
  const int d0 = 16 * NB * slab, dw = min(16 * NB, 2 * cs - d0);  // real columns of the slab
  double* wb = reinterpret_cast<double*>(f.wb[s] + w * (long)N * cs) + d0;
  double* t0 = reinterpret_cast<double*>(f.t0 + w * (long)N * ct + (s ? f.c[0] : 0)) + d0;
  const double2* V = f.vhs + w * 256L * R * R + lane;
  const double* E = f.e[s];

  // row blocks of this wave, and its column-split blocks of the last rows
  const int base = R / NWAVE, rem = R % NWAVE;
  const bool four = rem >= 4;
  const int nmain = base + (four && wave < 4 ? 1 : 0);
  const int r0 = base * NWAVE + (four ? 4 : 0), nx = (R - r0) * NB;
  int rb[MB + XB], xc[XB + 1];
  bool on[MB + XB];
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    on[m] = m < nmain;
    rb[m] = min(m * NWAVE + wave, R - 1);
  }
#pragma unroll
  for (int e = 0; e < XB; ++e) {
    const int x = ((wave + 4) & 7) + NWAVE * e;
    on[MB + e] = x < nx;
    rb[MB + e] = on[MB + e] ? r0 + x / NB : 0;
    xc[e] = on[MB + e] ? x % NB : 0;
  }

  for (int e = tid; e < 16 * R * LDP; e += NT) {
    const int r = e / LDP, d = e - r * LDP;
    P[e] = r < N && d < dw ? wb[(long)r * 2 * cs + d] : 0.0;
  }
  __syncthreads();

  v4d acc[MB][NB], ax[XB + 1];
  const unsigned neg = (c16 & 1) ? 0u : 0x80000000u;  // sign of B' at this column
  // accumulators <- A P; VH: A = VHS, else A = E
  auto product = [&](auto vh) {
    constexpr bool VH = decltype(vh)::value;
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[m][j] = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int e = 0; e < XB; ++e) ax[e] = v4d{0.0, 0.0, 0.0, 0.0};
    // Fragments of the 8-deep step `step` (k = 16 kb + 4 q + 2 h + t).  Every
    // wave loads for all its slots, an unused one the same block again: with
    // loads in branches the compiler cannot count them and waits for all.
    struct Frag {
      double2 x[MB + XB][2];
    };
    auto fetch = [&](Frag& F, int step) {
      const int kb = step >> 1, h = step & 1;
#pragma unroll
      for (int m = 0; m < MB + XB; ++m) {
        const int ib = rb[m], k = on[m] ? kb : 0, hh = on[m] ? h : 0;
        if (VH) {
          const double2* src = V + 256L * (ib * R + k) + 128 * hh;
          F.x[m][0] = src[0];
          F.x[m][1] = src[64];
        } else {
          const double* src = E + 256L * (ib * R + k) + 128 * hh + lane;
          F.x[m][0].x = src[0];
          F.x[m][1].x = src[64];
        }
      }
    };
    auto swapped = [&](double b) {
      const long long v = __double_as_longlong(swap_pair(b));
      return __longlong_as_double(v ^ ((long long)(unsigned long long)neg << 32));
    };
    auto multiply = [&](const Frag& F, int step) {
      const double* B = P + (16 * (step >> 1) + 4 * q + 2 * (step & 1)) * LDP + c16;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        double b[NB], xb[XB + 1];
#pragma unroll
        for (int j = 0; j < NB; ++j) b[j] = B[t * LDP + 16 * j];
#pragma unroll
        for (int e = 0; e < XB; ++e) xb[e] = B[t * LDP + 16 * xc[e]];
#pragma unroll
        for (int m = 0; m < MB; ++m)
          if (on[m]) {
#pragma unroll
            for (int j = 0; j < NB; ++j) acc[m][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(F.x[m][t].x, b[j], acc[m][j], 0, 0, 0);
            if (VH) {
#pragma unroll
              for (int j = 0; j < NB; ++j)
                acc[m][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(F.x[m][t].y, swapped(b[j]), acc[m][j], 0, 0, 0);
            }
          }
#pragma unroll
        for (int e = 0; e < XB; ++e)
          if (on[MB + e]) {
            ax[e] = __builtin_amdgcn_mfma_f64_16x16x4f64(F.x[MB + e][t].x, xb[e], ax[e], 0, 0, 0);
            if (VH) ax[e] = __builtin_amdgcn_mfma_f64_16x16x4f64(F.x[MB + e][t].y, swapped(xb[e]), ax[e], 0, 0, 0);
          }
      }
    };
    Frag f0, f1;
    fetch(f0, 0);
    for (int step = 0; step < 2 * R; step += 2) {
      fetch(f1, step + 1);
      multiply(f0, step);
      fetch(f0, min(step + 2, 2 * R - 1));
      multiply(f1, step + 1);
    }
  };
  // every accumulator block: fn(block, row block, column block)
  auto each = [&](auto fn) {
#pragma unroll
    for (int m = 0; m < MB; ++m)
      if (on[m]) {
#pragma unroll
        for (int j = 0; j < NB; ++j) fn(acc[m][j], rb[m], j);
      }
#pragma unroll
    for (int e = 0; e < XB; ++e)
      if (on[MB + e]) fn(ax[e], rb[MB + e], xc[e]);
  };
  // element v of a block: row 16 rb + q + 4 v, column 16 j + c16
  auto to_lds = [&] {
    __syncthreads();  // every wave is done reading the panel
    each([&](v4d& x, int r, int j) {
#pragma unroll
      for (int v = 0; v < 4; ++v) P[(16 * r + q + 4 * v) * LDP + 16 * j + c16] = x[v];
    });
    __syncthreads();
  };

  product(std::false_type{});
  each([&](v4d& x, int r, int j) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = 16 * r + q + 4 * v, d = 16 * j + c16;
      if (row < N && d < dw) t0[(long)row * 2 * ct + d] = x[v];
    }
  });
  to_lds();
  for (int n = f.nterms - 1; n >= 1; --n) {
    product(std::true_type{});
    const double sc = 1.0 / n;
    each([&](v4d& x, int r, int j) {
      const int d = 16 * j + c16;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = 16 * r + q + 4 * v;
        const double t = row < N && d < dw ? t0[(long)row * 2 * ct + d] : 0.0;
        x[v] = fma(sc, x[v], t);
      }
    });
    to_lds();
  }
  product(std::false_type{});
  each([&](v4d& x, int r, int j) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = 16 * r + q + 4 * v, d = 16 * j + c16;
      if (row < N && d < dw) wb[(long)row * 2 * cs + d] = x[v];
    }
  });
}

// E (N x N, row-major) -> [row block][k block][k % 4][k / 4][row], zero past N
__global__ void pack_e_kernel(const double* __restrict__ e, int N, int R, double* __restrict__ out) {
  const long t = blockIdx.x * 256L + threadIdx.x;
  if (t >= 256L * R * R) return;
  const int b = (int)(t >> 8), i = 16 * (b / R) + (int)(t & 15);
  const int k = 16 * (b % R) + 4 * (int)((t >> 4) & 3) + (int)((t >> 6) & 3);
  out[t] = i < N && k < N ? e[(long)i * N + k] : 0.0;
}

int blocks_of(int N) { return (N + 15) / 16; }

// Accumulator blocks a wave may hold: MB row blocks by NB column blocks.
bool held(int MB, int NB) { return MB >= 1 && MB <= 4 && NB >= 1 && NB <= 5 && MB * NB <= 10; }

int main_blocks(int R) { return R / NWAVE + (R % NWAVE >= 4 ? 1 : 0); }

// Blocks of the busiest SIMD of a work-group.
int simd_blocks(int R, int NB) {
  const int rem = R % NWAVE, base = 2 * (R / NWAVE) + (rem >= 4 ? 1 : 0), left = rem % 4;
  return base * NB + (left * NB + 3) / 4;
}

template <int MB, int NB, int XB>
int launch(const TrotArgs& a, long grid, size_t bytes, hipStream_t st) {
  static std::atomic<uint64_t> raised{0};
  AFQ_TRY(raise_lds(reinterpret_cast<const void*>(trot_f64_kernel<MB, NB, XB>), kLdsMax, raised, "propagator"));
  hipLaunchKernelGGL((trot_f64_kernel<MB, NB, XB>), dim3((unsigned)grid), dim3(NT), bytes, st, a);
  return launch_status("trot_f64_kernel");
}

}  // namespace

bool trot_f64_supported(int N) {
  const int R = blocks_of(N), MB = std::max(1, main_blocks(R));
  return held(MB, 1) && 16L * R * 16 * 8 <= kLdsMax;
}
long trot_f64_e_elems(int N) { return 256L * blocks_of(N) * blocks_of(N); }

int k_pack_e_f64(const double* e, int N, double* out, hipStream_t st) {
  const int R = blocks_of(N);
  hipLaunchKernelGGL(pack_e_kernel, dim3((unsigned)(R * R)), dim3(256), 0, st, e, N, R, out);
  return launch_status("pack_e_kernel");
}

int trot_f64(const TrotF64& f, hipStream_t st) {
  TrotArgs a{};
  a.f = f;
  a.R = blocks_of(f.N);
  const int MB = std::max(1, main_blocks(a.R));
  // Column blocks a slab: the least work of the busiest CU's work-groups, however
  // many of them share it; at equal work the larger slab, which reads the VHS
  // less often (N=100, 20 columns, 256 walkers: 3 blocks 87 us, 1 block 93, 2
  // blocks, which would fill two work-groups a CU, 101; N=150, 50 + 48 columns, 64
  // walkers: 4 blocks 192, 2 blocks 188).
  int NB = 0;
  double best = 0.0;
  for (int nb = 1; nb <= 5; ++nb) {
    const long lds = 16L * a.R * 16 * nb * 8;
    if (!held(MB, nb) || lds > kLdsMax) continue;
    long S = 0;
    for (int s = 0; s < f.nspin; ++s) S += ((f.c[s] + 7) / 8 + nb - 1) / nb;
    const double t = std::ceil((double)(S * f.W) / 256.0) * simd_blocks(a.R, nb);
    if (NB == 0 || t <= best) {
      NB = nb;
      best = t;
    }
  }
  if (NB == 0) return fail(AFQ_E_UNSUPPORTED, "fused FP64 propagator: norb too large");
  long S = 0;
  for (int s = 0; s < f.nspin; ++s) S += a.nslab[s] = ((f.c[s] + 7) / 8 + NB - 1) / NB;
  const long grid = 8L * ((f.W + 7) / 8) * S;
  if (grid > 0x7fffffffL) return fail(AFQ_E_UNSUPPORTED, "fused FP64 propagator: grid too large");
  const size_t bytes = 16L * a.R * 16 * NB * 8;
  const int XB = ((a.R % NWAVE % 4) * NB + NWAVE - 1) / NWAVE;  // 0, 1 or, from NB = 3, 2
#define TROT(mb, nb)                                       \
  if (MB == mb && NB == nb)                                \
  return XB == 0   ? launch<mb, nb, 0>(a, grid, bytes, st) \
         : XB == 1 ? launch<mb, nb, 1>(a, grid, bytes, st) \
                   : launch<mb, nb, (nb > 2 ? 2 : 1)>(a, grid, bytes, st)
  TROT(1, 1);
  TROT(1, 2);
  TROT(1, 3);
  TROT(1, 4);
  TROT(1, 5);
  TROT(2, 1);
  TROT(2, 2);
  TROT(2, 3);
  TROT(2, 4);
  TROT(2, 5);
  TROT(3, 1);
  TROT(3, 2);
  TROT(3, 3);
  TROT(4, 1);
  TROT(4, 2);
#undef TROT
  return fail(AFQ_E_UNSUPPORTED, "fused FP64 propagator: no tile");
}

}  // namespace afq

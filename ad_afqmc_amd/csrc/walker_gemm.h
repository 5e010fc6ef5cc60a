// The two FP64 products of a step over all walkers at once (walker_gemm.hip).
#pragma once
#include "afq_internal.h"

namespace afq {

// Force bias: out (W, G) = fac sum_s G_s (W, K_s) . rot_chol_s^T (K_s, G).
struct ForceBias64 {
  int W = 0, G = 0, nspin = 1;
  long K[2] = {0, 0};
  const double2* green[2] = {nullptr, nullptr};
  const double* rc[2] = {nullptr, nullptr};
  double fac = 1.0;
  double2* out = nullptr;
  double* ws = nullptr;  // partial sums
  long ws_elems = 0;
};
// doubles of workspace a force bias of these sizes can use
long force_bias_f64_ws(int W, int G, long K0, long K1);
int force_bias_f64(const ForceBias64& f, hipStream_t st);

// VHS of symmetric Cholesky vectors, i sqrt(dt) x (W, G) . L (G, npk), written
// by 16 x 16 orbital blocks of the full matrix in the order the propagator's
// fragments read them: block (ib, kb) of R x R, then [k % 4][k / 4][row].
long vhs_f64_elems(int N);  // complex elements a walker
int vhs_f64(const double2* xs, const double* lp, int N, int G, int W, double sqdt, double2* out, hipStream_t st);

}  // namespace afq

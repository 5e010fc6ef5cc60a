// Fused FP64 propagator (trot_f64.hip).
#pragma once
#include "afq_internal.h"

namespace afq {

struct TrotF64 {
  int N = 0, W = 0, nspin = 1, nterms = 1;
  int c[2] = {0, 0};                       // columns of each walker buffer
  double2* wb[2] = {nullptr, nullptr};     // (W, N, c), in place
  const double* e[2] = {nullptr, nullptr}; // packed exp(-dt/2 h1)
  const double2* vhs = nullptr;            // the blocks of vhs_f64
  double2* t0 = nullptr;                   // scratch, (W, N, c[0] + c[1])
};
bool trot_f64_supported(int N);
// doubles of the packed exp(-dt/2 h1), and the packing
long trot_f64_e_elems(int N);
int k_pack_e_f64(const double* e, int N, double* out, hipStream_t st);
int trot_f64(const TrotF64& f, hipStream_t st);

}  // namespace afq

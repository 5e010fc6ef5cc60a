// FP64 exchange over the unoccupied orbitals of the trial (exchange_f64.hip).
#pragma once
#include "afq_internal.h"

namespace afq {

constexpr int kExchangeF64MaxO = 128;

// Work-group tile: WR x WC waves of MB x NB MFMA blocks hold gw g's of wn walkers.
struct ExF64Tile {
  int MB, NB, WR, WC, gw, wn;
};
ExF64Tile exchange_f64_tile(int O);
// The tile for W walkers: the same rows, fewer columns where walkers are few.
ExF64Tile exchange_f64_tile(int O, int W, int G);
int exchange_f64_nchunk(int O, int G);
// Partial K's of a walker, at most.
int exchange_f64_slots(int O, int N, int G);
// Few walkers: exchange_f64_theta, once for both spins, fills the packed theta and
// the partial K's of it before k_exchange_f64 (green null); with ene1 (not null)
// also the one-body energies of all spins, each times fac.
bool exchange_f64_few(int O, int N, int W);
long exchange_f64_most_few(int O, int N);  // the most walkers that are few
struct ExTheta {
  const double2* green;
  const double *Q, *mt, *k0, *rh1;
  int O;
  double2* thetap;
  double2* kpart;
};
int exchange_f64_theta(const ExTheta* sets, int nsets, int N, int G, int W, double fac, double2* ene1,
                       hipStream_t st);

struct ExF64 {
  const double* a;        // packed rot_chol Q
  const double2* theta;   // packed slabs of B (pack_b_kernel)
  const double* c0;       // (G,) tr f0_g
  int O, Nv, n8, G, W, gw, wn, nwg, nchunk, kstride, cpg, gp, strip;
  long T8, lds_elems;
  double2* coul;          // (W, G)
  double2* kpart;         // (W, kstride)
};

// Sizes of the packed rot_chol Q (doubles), of the packed theta (complex) and
// of the setup workspace (doubles, for two spins of O).
long exchange_f64_a_elems(int O, int N, int G);
long exchange_f64_b_elems(int O, int N, int W);
long exchange_f64_tmp_elems(int O, int N, int G);
// Per trial of up to two spins: Q (N, N - O), orthonormal complement of span(mo),
// and P (N, O) = mo (mo^T mo)^-1.  tmp: the setup workspace of the larger one.
struct ExTrial {
  const double* mo;
  int O;
  double* Q;
  double* P;
};
int exchange_f64_set_trial(const ExTrial* sets, int nsets, int N, double* tmp, hipStream_t st);
// From rot_chol (G, O, N) of up to two spins: a, c0 (G,), mt (O, N - O), k0 (1,);
// kg (2 G,) scratch.
struct ExChol {
  const double *rc, *Q, *P;
  int O;
  double *a, *c0, *mt, *k0;
};
int exchange_f64_set_chol(const ExChol* sets, int nsets, int N, int G, double* kg, double* tmp, double* ws,
                          long ws_elems, hipStream_t st);
// Rows (k pairs) of the packed theta of one walker group.
int exchange_f64_npairs(int Nv);
// green null: thetap and the last partial K's are filled already.
// c_g (W, G) and the *nch_out partial K's of every walker; theta (W, O, N - O) and
// thetap (exchange_f64_b_elems) are scratch.
int k_exchange_f64(const double* a, const double* Q, const double* c0, const double* mt, const double* k0,
                   const double2* green, double2* theta, double2* thetap, int O, int N, int G, int W, double2* coul,
                   double2* kpart, int* nch_out, hipStream_t st);

}  // namespace afq

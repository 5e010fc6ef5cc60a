// One work-group per walker for small FP64 jobs (small.hip).
#pragma once
#include "afq_internal.h"

namespace afq {

// Limits of the walkers a work-group holds: orbitals in a step, and occupied
// orbitals per spin (one wave's Gauss-Jordan panel).
constexpr int kSmallMaxN = 48, kSmallMaxO = 16;

// nspin: spins measured; spin s is columns off[s] .. off[s] + occ[s] of the
// N x c panel.  nbuf walker buffers of cb[b] columns fill the panel one after
// another.
struct SmallJob {
  int N, G, W, nspin, nbuf, c;
  int occ[2], off[2], cb[2];
  double2* wbuf[2];
  const double* mo[2];
  double2* Sinv[2];
  double2* det[2];
};

struct SmallStep {
  SmallJob b;
  const double* ex[2];    // exp(-dt/2 h1) of each walker buffer
  const double2* lt;      // packed L and rot_chol (k_small_pack_l, k_small_pack_rc)
  const double2* rcp;
  int sym, nterms, nsteps;
  double fac, dt;         // force-bias factor
  const double2* mf;
  const double* fields;   // (nsteps, W, G)
  const double2* h0p;
  const double* scalars;  // the shift that the steps start with
  double* h;              // (nsteps, W): the phaseless factor at that shift, not clipped
  double2* overlaps;      // in: of the incoming walkers; out: of the new ones
  // of the last step
  double2 *fb, *xs, *terms, *ov_new;
};

struct SmallMeasure {
  SmallJob b;
  int qr, inverse, energy;  // inverse: also S^-1 and the Green's functions
  double fac;             // one-body factor
  double2* overlaps;      // may be null
  double2* green[2];
  const double* rh1[2];
  double2* ene1;
  // exchange operands of every spin (exchange_f64.hip): theta packed, and the
  // walker-independent part of K
  const double* q[2];
  const double* mt[2];
  const double* k0[2];
  double2* thetap[2];     // null: left to the exchange (exchange_f64_few)
  double2* kpart[2];
  int wn[2], c2[2], npr[2], nchunk[2];
  // or, with `whole`, the exchange and the energy here (small_energy_whole)
  int whole;
  const double* rc[2];
  double h0;
  double2* energies;
};

// Whether a walker's exchange is little enough for its own work-group.
bool small_energy_whole(int N, int G, int occ0, int occ1);

// L and rot_chol as the step reads them, by Cholesky index: L's entries (i, j),
// i >= j, row by row where L_g is symmetric (else all), and the flattened
// rot_chol of every measured spin, both padded to pairs.
long small_l_pairs(int N, bool sym);
long small_rc_pairs(int N, int osum);
int k_small_pack_l(const double* chol, int N, int G, bool sym, double2* out, hipStream_t st);
int k_small_pack_rc(const double* rc0, int n0, const double* rc1, int n1, int G, double2* out, hipStream_t st);
// LDS bytes of a step's and of a measurement's work-group; 0 if the sizes are
// past the limits.
size_t small_step_lds(int N, int G, int c, int osum, int nbuf);
size_t small_measure_lds(int N, int c, int osum, int nspin);
// Whether a phaseless step of W walkers is better off in one work-group per
// walker, which reads L and rot_chol for every walker, than in batched products.
bool small_step_pays(int N, int G, int osum, int W, bool sym);
int k_small_measure(const SmallMeasure& p, hipStream_t st);
// nsteps phaseless steps of every walker; a walker's path does not depend on
// the weights, which k_small_weights then takes through the steps.
int k_small_step(const SmallStep& p, hipStream_t st);
int k_small_weights(const double* h, int nsteps, int W, double dt, double* weights, double* scalars, hipStream_t st);

}  // namespace afq

// sfx_chain1d.h -- several ranks of a chain on a 1-D lattice in one launch
// (FP64, unscaled, full store; sfx_chain1d.hip).
#pragma once

#include "sfx_kernels.h"

namespace sfx {

constexpr int kChain1MaxSites = 4000;  // two LDS rank buffers stay below 64 KiB

// one rank step: next = g * stencil(current); stored to out (may be null);
// acc += next * pair when acc is set
struct Chain1Step {
  const double* g;
  double* out;
  const double* pair;
  double* acc;
};

bool chain1d_ok(const DevLattice& L);
// advances the rank in0 through steps[0..n) (a device array); the final rank
// goes to last (may be null)
void launch_chain1d(const DevLattice& L, const double* in0, const Chain1Step* steps, int n, double* last,
                    hipStream_t st);

// a run of consecutive ranks of one state, and a molecule as k_scf1d sees it
struct Chain1Run {
  int state, count;
};
struct Chain1Mol {
  int index, N, freedom, kind;
  int run0, nruns;  // its runs, in rank order
  unsigned uses;
  int lo, hi;       // range_restricted: the box
  double phib, theta, phi_range;
};

// arrays of a 1-D system as System holds them
struct Scf1Args {
  SysParams sp;
  unsigned shared;        // states of more than one molecule
  Chain1Mol mols[SFX_MAXM];  // in the order of evaluation
  const Chain1Run* runs;
  int nruns;
  SiteVec x;
  double* u;              // may be null: x's copy in the internal layout
  const unsigned char* itmask;
  const double* fprof;
  double* swf;
  float* swf32;
  double *store, *phi_m, *phi, *rho, *phitot, *molscal, *phib_state, *cbulk;
  SiteOut f;              // may be null: phi only
  // tangent
  int base;               // with the base evaluation
  SiteVec v;
  double *dstore, *dphi_m;
  SiteOut jv;
};

// one workgroup evaluates the whole system (up to 1024 layers whose arrays fit LDS)
bool scf1d_ok(const DevLattice& L, int ns, bool tangent);
void launch_scf1d(const DevLattice& L, const Scf1Args& a, bool tangent, hipStream_t st);

}  // namespace sfx

// sfx_close.h -- the launches that close an evaluation or a Jacobian product
// after the propagator sweeps (sfx_close.hip).
#pragma once

#include "sfx_kernels.h"

namespace sfx {

constexpr int kEndBlocks = 256;  // workgroups of an end sum per molecule: one per CU

// End rank of a molecule: its weighted sum (ComputeLnGN before the log) gives
// the molecule's scalars, that of its tangent the tangent scalars.
struct EndMol {
  MolParams mp;
  const void* G;      // T, or double for a monomer (its SWF); second order: six components
  const void* dG;     // tangent, of the same type; for a monomer the direction v (dG = -v g)
  const double* lnf;  // FP32: log scale of the end rank; nullptr: unscaled, MS_REF becomes 0
  bool f32, unscaled;
  // FP32 by blocked launches: step maxima of the chains' last ranks that no
  // launch reads, and the word set when one is below kLowMax (null: not by blocked
  // launches; with it G and the maxima carry kBlockScale)
  const unsigned* endmax[2];
  unsigned* low;
};
struct EndArgs {
  int n;  // entries; a solvent may only close on entries before it or finished molecules
  EndMol e[SFX_MAXM];
  int nm;
  double* molscal;   // written with `base`, else read
  double* dmol;      // with `tangent`
  double* partial;   // [2][SFX_MAXM][kEndBlocks]
  unsigned* ticket;  // 0 before and after
  bool base, tangent;
};
void launch_end_sums(const DevLattice& L, const EndArgs& a, hipStream_t st);

// phi_m of the molecules from their accumulators, the state totals and bulk
// fractions (base) and their tangents (tangent)
enum { CLOSE_DONE = 0, CLOSE_CHAIN, CLOSE_MONOMER };  // CLOSE_DONE: phi_m is there
struct PhiArgs {
  int nm, ns;
  unsigned uses[SFX_MAXM];
  int mode[SFX_MAXM];
  int two[SFX_MAXM];  // a second accumulator (middle-out sweeps)
  int frozen[SFX_MAXS];
  const void *acc, *acc2, *dacc, *dacc2;  // T, [m][state][M]
  const double *swf, *fprof, *vdir;       // vdir: per-state direction
  const double *molscal, *dmol;
  double *phi_m, *phi, *dphi;
  double *phib_state, *cbulk;
  bool base, tangent;
};
template <typename T>
void launch_phi_close(const DevLattice& L, const SysParams& sp, const PhiArgs& a, hipStream_t st);

// contact averages and total of phi (base), the residual (f), the linearised residual (jv)
struct FieldArgs {
  const unsigned char* itmask;
  const double *swf, *phi, *cbulk;
  double *rho, *phitot;
  SiteOut f;                   // p null: contact averages alone
  SiteVec v;                   // jv: direction and tangents
  const double *dphi, *dmol;
  double* drho;
  SiteOut jv;                  // p null: no product
  bool base;
};
void launch_field_close(const DevLattice& L, const SysParams& sp, const FieldArgs& a, hipStream_t st);

}  // namespace sfx

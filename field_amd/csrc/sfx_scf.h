// sfx_scf.h -- the arithmetic of one site, one molecule and one system, shared
// by the kernels that run it launch by launch over a whole lattice and by the
// one that runs a 1-D system in a single workgroup (sfx_chain1d.hip): both give
// the same bits, but for a product's last operations, which the compiler fuses
// in each as it finds them.
#pragma once

#include "sfx_device.h"
#include "sfx_kernels.h"

namespace sfx {

// Molecule scalars after a sweep from the weighted sum s of its end rank (one
// thread). Normalisation per freedom: SF_Monomer1stO.cpp:110-130,
// SF_Homopol1stO.cpp:599-619, SF_Copol1stO.cpp:1242-1275. phib_of(m): the bulk
// fraction of another molecule. The accumulators carry exp(-ref) 2^power.
template <class PhibOf>
__device__ __forceinline__ void mol_scalars(const MolParams& mp, double s, double lnscale, double ref, int power,
                                            int nmol, PhibOf&& phib_of, double* scal) {
  const double lnsum = mp.kind == 3 ? log(s / 6.0) : log(s);  // second order: Lat3D2ndO.cpp:1024
  const double lnGN = lnsum + lnscale;                        // FP32: plus the log-scale of the final rank
  const double N = mp.N;
  double phib = mp.phib, lnC, lnpref;
  if (mp.freedom == SFX_SOLVENT) {
    phib = 1.0;
    for (int m = 0; m < nmol; m++)
      if (m != mp.index) phib -= phib_of(m);
  }
  // half-stored chains (SymMatrix1 factor 2); second order divides by 6 (Lat3D2ndO.cpp:1037)
  const double f = mp.kind == 2 ? 2.0 : mp.kind == 3 ? 1.0 / 6.0 : 1.0;
  double pref;
  if (mp.freedom == SFX_RANGE_RESTRICTED) {
    // the profile before the range condition fixes its constant (range_scalars)
    lnC = 0.0;
    phib = 0.0;
    pref = f * exp(ref);
  } else if (mp.freedom == SFX_RESTRICTED) {
    lnC = log(mp.theta) - lnGN - (mp.kind == 0 ? 0.0 : log(N));
    phib = mp.theta / exp(lnGN);
    lnpref = lnC;
    pref = f * exp(lnpref + ref);
  } else {
    // phi = (phi_b / N) G G_inv / g: phi_b multiplies directly, since the
    // solvent closure can make it negative (NormPhiFree, Lat1DFlat1stO.cpp:317-331)
    const double C = mp.kind == 0 ? phib : phib / N;
    lnC = log(C);  // NaN for phi_b <= 0, as ln of the reference's lnCb; used by the free energy only
    pref = f * C * exp(ref);
  }
  scal[MS_LNGN] = lnGN;
  scal[MS_LNC] = lnC;
  scal[MS_PHIB] = phib;
  scal[MS_PREF] = ldexp(pref, -power);
}

// range_restricted: the constant from the profile's sum s over the box, after mol_scalars
__device__ __forceinline__ void range_scalars(double s, double phi_range, int N, double* scal) {
  const double C = phi_range / s;
  scal[MS_RANGE_C] = C;
  scal[MS_PREF] *= C;
  scal[MS_LNC] = log(C);
  // theta = sum_z L phi = C N G_N (every rank composes to G_N), so phi_b = theta / G_N = N C
  scal[MS_PHIB] = (double)N * C;
}

// phi of a molecule at a site from its accumulator(s)
__device__ __forceinline__ double phi_site(double acc, double g, double pref) {
  return g > 0 ? (acc / g) * pref : 0.0;
}

// segment bulk fractions and ChemIntBulk (SF_MolStructure.cpp:605-612,
// SF_SegmentList.cpp:610-623) by one wave, a lane per state; cb: ChemIntBulk in
// LDS as well
__device__ __forceinline__ void bulk_fractions_wave(const SysParams& sp, const double* molscal, double* phib_state,
                                                    double* cbulk, double* cb) {
  const int t = (int)threadIdx.x & 63;
  const bool in = t < sp.ns;
  double pb = 0;
  if (in) {
    if (sp.melt)
      pb = sp.melt_phib[t];
    else if (!sp.frozen[t])
      for (int m = 0; m < sp.nm; m++) pb += molscal[m * MS_COUNT + MS_PHIB] * sp.mol_frac[m * SFX_MAXS + t];
    phib_state[t] = pb;
  }
  double c = 0;
  for (int j = 0; j < sp.ns; j++) {
    const double pj = __shfl(pb, j, 64);
    const double x = in && !sp.frozen[t] ? sp.chi[t * SFX_MAXS + j] : 0.0;
    if (x != 0) c += x * pj;
  }
  if (in) cbulk[t] = cb[t] = c;
}

// f = -1 + 1/phitot + u'_i - <u'> of one iteration site (SF_Solve.cpp:554-590):
// swf(t), rho(t): the site's SWF and contact average of state t; put(k, f).
// NS: a bound on the states and iteration variables; below SFX_MAXS the loops
// unroll, for averages in registers
template <int NS = SFX_MAXS, class Swf, class Rho, class Put>
__device__ __forceinline__ void residual_site(const SysParams& sp, double pt, const double* cbulk, Swf&& swf,
                                              Rho&& rho, Put&& put) {
  const int nv = sp.n_itvar;
  constexpr int unroll = NS < SFX_MAXS ? NS : 1;
  double up[NS];
  double av = 0;
#pragma unroll unroll
  for (int k = 0; k < NS; k++) {
    if (k >= nv) break;
    int t = sp.itvar_rep[k];
    double ci = 0;
#pragma unroll unroll
    for (int j = 0; j < NS; j++) {
      if (j >= sp.ns) break;
      double x = sp.chi[t * SFX_MAXS + j];
      if (x != 0) ci += x * rho(j);
    }
    double v = -log(swf(t));
    v -= ci / pt;
    v += cbulk[t];
    up[k] = v;
    av += v;
  }
  av /= nv;
#pragma unroll unroll
  for (int k = 0; k < NS; k++) {
    if (k >= nv) break;
    put(k, -1.0 + 1.0 / pt + up[k] - av);
  }
}

// tangent molecule scalars from the weighted sums s1 of the end rank and s2 of
// its tangent (any = false: no sums): d[0] = dlnGN, d[1] = dpref/pref,
// d[2] = dphib, d[3] the prefactor of the sweep's own scaling
template <class DphibOf>
__device__ __forceinline__ void tmol_scalars(const MolParams& mp, bool any, double s1, double s2, const double* ms,
                                             int nmol, DphibOf&& dphib_of, double* d) {
  const double dln = any ? s2 / s1 : 0.0;
  const double phib = ms[MS_PHIB];
  const double f = mp.kind == 2 ? 2.0 : mp.kind == 3 ? 1.0 / 6.0 : 1.0;
  if (mp.freedom == SFX_RESTRICTED)
    d[3] = f * exp(log(mp.theta) - ms[MS_LNGN] - (mp.kind == 0 ? 0.0 : log((double)mp.N)) + ms[MS_REF]);
  else
    d[3] = f * (mp.kind == 0 ? phib : phib / mp.N) * exp(ms[MS_REF]);
  d[3] = ldexp(d[3], -(int)ms[MS_POW]);
  d[0] = dln;
  if (mp.freedom == SFX_RESTRICTED) {
    d[1] = -dln;
    d[2] = -phib * dln;
  } else if (mp.freedom == SFX_SOLVENT) {
    double dpb = 0;
    for (int m = 0; m < nmol; m++)
      if (m != mp.index) dpb -= dphib_of(m);
    d[2] = dpb;
    d[1] = phib != 0 ? dpb / phib : 0.0;
  } else {
    d[1] = 0;
    d[2] = 0;
  }
}

// dphi of a molecule at a site: phi, SWF, direction and tangent accumulator there
__device__ __forceinline__ double tphi_site(bool monomer, double phi, double g, double v, double dacc,
                                            const double* dm) {
  const double rel = dm[1];
  if (monomer) return phi * (rel - v);
  return g > 0 ? phi * (rel + v) + dm[3] * dacc / g : 0.0;
}

// linearised residual of one iteration site (SF_Solve.cpp:554-590): v(k) the
// direction, rho/drho(t) contact averages, pt/dpt the totals, dmol the tangent
// molecule scalars; put(k, jv)
template <int NS = SFX_MAXS, class V, class Rho, class Drho, class Put>
__device__ __forceinline__ void jres_site(const SysParams& sp, double pt, double dpt, const double* dmol, V&& v,
                                          Rho&& rho, Drho&& drho, Put&& put) {
  const int nv = sp.n_itvar;
  constexpr int unroll = NS < SFX_MAXS ? NS : 1;
  double du[NS];
  double av = 0;
#pragma unroll unroll
  for (int k = 0; k < NS; k++) {
    if (k >= nv) break;
    int t = sp.itvar_rep[k];
    double ci = 0, dci = 0, dcb = 0;
#pragma unroll unroll
    for (int j = 0; j < NS; j++) {
      if (j >= sp.ns) break;
      double c = sp.chi[t * SFX_MAXS + j];
      if (c == 0) continue;
      ci += c * rho(j);
      dci += c * drho(j);
      if (!sp.melt && !sp.frozen[j]) {
        double dpb = 0;
        for (int m = 0; m < sp.nm; m++) dpb += dmol[m * 4 + 2] * sp.mol_frac[m * SFX_MAXS + j];
        dcb += c * dpb;
      }
    }
    double d = v(k) - dci / pt + ci * dpt / (pt * pt) + dcb;
    du[k] = d;
    av += d;
  }
  av /= nv;
#pragma unroll unroll
  for (int k = 0; k < NS; k++) {
    if (k >= nv) break;
    put(k, -dpt / (pt * pt) + du[k] - av);
  }
}

// one rank of a tangent chain and one term of its composition; the products are
// contracted as written, so every kernel that uses them gives the same bits
template <typename T>
__device__ __forceinline__ T tan_step(T da, T v, T a) {  // (A[dG] - v A[G]); times g
  return fma(-v, a, da);
}
template <typename T>
__device__ __forceinline__ T tan_compose(T dG, T Gp, T G, T dGp) {  // dG Gp + G dGp
  return fma(dG, Gp, G * dGp);
}

// contact averages of one site, halo sites that are not surfaces excluded
// (SetBoundaries fills those)
__device__ __forceinline__ bool has_side(const DevLattice& L, int x, int y, int z) {
  if (is_interior(L, x, y, z)) return true;
  const int c[3] = {x, y, z}, n[3] = {L.nx, L.ny, L.nz};
  for (int k = 0; k < L.grad; k++)
    if ((c[k] == 0 && L.surf1[k]) || (c[k] == n[k] + 1 && L.surf2[k])) return true;
  return false;
}

}  // namespace sfx

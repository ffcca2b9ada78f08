// sfx_close.hip -- what follows the propagator sweeps of an evaluation or a
// Jacobian product: end sums and molecule scalars, volume fractions, contact
// averages and the (linearised) residual, in three launches.
//
// As a launch per molecule and quantity this was 11 to 15 launches, 40 us or
// more on any lattice. Every launch costs 2.5 us of dispatch and drain whatever
// it does, and a profile written by one is read again by the next. Together
// they take 18 us on the 64 x 128 pore (with them a residual went from 154 to 130
// us, a product from 217 to 178), 34 us for a product at 64^3 (327 to 300 us) and
// 103 us at 128^3, where 70 are the profiles' traffic (139 us before).
//   k_end_sums    every molecule's end sum; the workgroup that finishes last
//                 adds the partial sums in a fixed order and derives the
//                 scalars, which were a launch of one workgroup each
//   k_phi_close   phi_m, phi_t and their tangents, site by site
//   k_field_close contact averages and residuals; the averages stay in
//                 registers (up to four states) beside the copy the free
//                 energy and the transposed products read
#include "sfx_close.h"

#include <algorithm>

#include "sfx_device.h"
#include "sfx_scf.h"

namespace sfx {

constexpr int kCB = 256;

template <typename T, bool TAN>
__device__ __forceinline__ void end_terms(const DevLattice& L, const EndMol& e, const T* __restrict__ G,
                                          const T* __restrict__ dG, long long q, double& s, double& ds) {
  int x, y, z;
  interior_coords(L, q, x, y, z);
  const long long r = sidx(L, x, y, z);
  if (e.mp.kind == 3) {
    // flat 1-D sums every layer plainly (Lat1D2ndO.cpp ComputeLnGN); 2-D and 3-D
    // halve mirror2 edges (Lat2D2ndO.cpp:387-439, Lat3D2ndO.cpp:996-1025);
    // curved lattices weight by the layer volume (Lat1DCyl2ndO.cpp:319-330,
    // Lat2DCyl2ndO.cpp:410-462)
    const double w = L.grad == 1 && !L.curved ? 1.0 : lngn_weight(L, x, y, z);
    for (int k = 0; k < 6; k++) {
      s += (double)G[(long long)k * L.M + r] * w;
      if constexpr (TAN) ds += (double)dG[(long long)k * L.M + r] * w;
    }
    return;
  }
  const double w = lngn_weight(L, x, y, z);
  const double g = (double)G[r];
  s += g * w;
  if constexpr (TAN) ds += e.mp.kind == 0 ? -(double)dG[r] * g * w : (double)dG[r] * w;
}

template <typename T, bool TAN, int NT>
__device__ __forceinline__ void end_sum(const DevLattice& L, const EndMol& e, double& s, double& ds) {
  const T* const G = (const T*)e.G;
  const T* const dG = (const T*)e.dG;
  const long long stride = (long long)gridDim.x * NT;
#pragma unroll 2
  for (long long q = site_ordinal(); q < L.V; q += stride) end_terms<T, TAN>(L, e, G, dG, q, s, ds);
}

// grid (workgroups, entries). Bound by memory round trips one after the other:
// the sums, the ticket, the last workgroup's read of the others' partial sums.
// Those cross the XCDs' L2 caches as relaxed atomics of device scope, with a
// wait for the store before the ticket: a __threadfence() writes the whole L2
// back, once per workgroup (18 us instead of 12 for a product at 64^3). What the
// scalars need besides is loaded before the sums.
template <bool TAN, int NT>
__global__ void __launch_bounds__(NT) k_end_sums(DevLattice L, EndArgs a) {
  const EndMol& e = a.e[blockIdx.y];
  __shared__ double r1[NT / 64], r2[NT / 64], s1[SFX_MAXM], s2[SFX_MAXM];
  __shared__ double ph[SFX_MAXM], dph[SFX_MAXM];
  __shared__ bool last;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  MolParams mp{};
  double sc[MS_COUNT] = {}, lnf = 0;
  if (t < a.n) {
    const EndMol& m = a.e[t];
    mp = m.mp;
    if (m.lnf) lnf = *m.lnf;
    const double* const old = a.molscal + mp.index * MS_COUNT;
    if (!m.unscaled) {
      sc[MS_REF] = old[MS_REF];
      sc[MS_POW] = old[MS_POW];
    }
    if (!a.base) {
      sc[MS_LNGN] = old[MS_LNGN];
      sc[MS_PHIB] = old[MS_PHIB];
    }
  }
  if (t < a.nm) {
    ph[t] = a.molscal[t * MS_COUNT + MS_PHIB];
    if constexpr (TAN) dph[t] = a.dmol[t * 4 + 2];
  }
  float em[2] = {kBlockScale, kBlockScale};
  const bool check = e.low && blockIdx.x == 0 && wave == 0;
  if (check)
    for (int k = 0; k < 2; k++)
      if (e.endmax[k]) em[k] = __uint_as_float(e.endmax[k][lane * kSlotStride]);
  double s = 0, ds = 0;
  if (e.f32)
    end_sum<float, TAN, NT>(L, e, s, ds);
  else
    end_sum<double, TAN, NT>(L, e, s, ds);
  for (int o = 32; o > 0; o >>= 1) {
    s += __shfl_xor(s, o, 64);
    if constexpr (TAN) ds += __shfl_xor(ds, o, 64);
  }
  if (check) {
    for (int o = 32; o > 0; o >>= 1) {
      em[0] = fmaxf(em[0], __shfl_xor(em[0], o, 64));
      em[1] = fmaxf(em[1], __shfl_xor(em[1], o, 64));
    }
    if (lane == 0 && !(fminf(em[0], em[1]) * kBlockDown >= kLowMax)) *e.low = 1u;
  }
  if (lane == 0) {
    r1[wave] = s;
    r2[wave] = ds;
  }
  __syncthreads();
  double* const p1 = a.partial;
  double* const p2 = a.partial + SFX_MAXM * kEndBlocks;
  if (t == 0) {
    s = ds = 0;
    for (int w = 0; w < NT / 64; w++) {
      s += r1[w];
      ds += r2[w];
    }
    const unsigned k = blockIdx.y * kEndBlocks + blockIdx.x;
    __hip_atomic_store(p1 + k, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if constexpr (TAN) __hip_atomic_store(p2 + k, ds, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the stores have arrived before the ticket
    const unsigned total = gridDim.x * gridDim.y;
    last = __hip_atomic_fetch_add(a.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == total - 1;
  }
  __syncthreads();
  if (!last) return;
  // a wave per entry, its partial sums in order
  for (int k = wave; k < a.n; k += NT / 64) {
    double u = 0, du = 0;
    for (int i = lane; i < (int)gridDim.x; i += 64) {
      u += __hip_atomic_load(p1 + k * kEndBlocks + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if constexpr (TAN) du += __hip_atomic_load(p2 + k * kEndBlocks + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    for (int o = 32; o > 0; o >>= 1) {
      u += __shfl_xor(u, o, 64);
      if constexpr (TAN) du += __shfl_xor(du, o, 64);
    }
    if (lane == 0) {
      s1[k] = u;
      s2[k] = du;
    }
  }
  if (t == 0) *a.ticket = 0u;
  __syncthreads();
  // a thread per molecule; the solvent, which closes on the others, last
  double* const out = a.molscal + mp.index * MS_COUNT;
  for (int pass = 0; pass < 2; pass++) {
    if (t < a.n && (mp.freedom == SFX_SOLVENT) == (pass == 1)) {
      if (a.base) {
        mol_scalars(mp, a.e[t].low ? s1[t] * kBlockDown : s1[t], lnf, sc[MS_REF], (int)sc[MS_POW], a.nm, [&](int o) { return ph[o]; }, sc);
        ph[mp.index] = sc[MS_PHIB];
        out[MS_LNGN] = sc[MS_LNGN];
        out[MS_LNC] = sc[MS_LNC];
        out[MS_PHIB] = sc[MS_PHIB];
        out[MS_PREF] = sc[MS_PREF];
      }
      out[MS_REF] = sc[MS_REF];
      out[MS_POW] = sc[MS_POW];
      if constexpr (TAN) {
        double d[4];
        tmol_scalars(mp, true, s1[t], s2[t], sc, a.nm, [&](int o) { return dph[o]; }, d);
        dph[mp.index] = d[2];
        for (int k = 0; k < 4; k++) a.dmol[mp.index * 4 + k] = d[k];
      }
    }
    __syncthreads();
  }
}

void launch_end_sums(const DevLattice& L, const EndArgs& a, hipStream_t st) {
  if (a.n == 0) return;
  SFX_REQUIRE(a.n <= SFX_MAXM, SFX_E_INVALID, "too many molecules to close");
  // at most kEndBlocks workgroups, however large the lattice: the last one reads
  // that many partial sums. From 65536 sites on they have 1024 threads, for
  // more loads in flight (128^3: 35 us with 256 threads)
  if (L.V > kEndBlocks * kCB) {
    const dim3 grid((unsigned)std::min<long long>(kEndBlocks, grid1(L.V, 1024)), (unsigned)a.n);
    if (a.tangent)
      k_end_sums<true, 1024><<<grid, 1024, 0, st>>>(L, a);
    else
      k_end_sums<false, 1024><<<grid, 1024, 0, st>>>(L, a);
  } else {
    const dim3 grid(grid1(L.V, kCB), (unsigned)a.n);
    if (a.tangent)
      k_end_sums<true, kCB><<<grid, kCB, 0, st>>>(L, a);
    else
      k_end_sums<false, kCB><<<grid, kCB, 0, st>>>(L, a);
  }
  SFX_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Grid (sites, states): bound by HBM on large lattices (every profile once), on
// small ones by the loads a thread waits for one after the other, which is why
// a state has threads of its own (three states in one thread: 7.5 us at 64 x
// 128). One workgroup more works out the bulk fractions.
template <typename T, bool BASE, bool TAN>
__global__ void __launch_bounds__(kCB) k_phi_close(DevLattice L, SysParams sp, PhiArgs a) {
  if constexpr (BASE) {
    if (blockIdx.x == gridDim.x - 1) {
      __shared__ double cb[SFX_MAXS];
      if (blockIdx.y == 0 && threadIdx.x < 64) bulk_fractions_wave(sp, a.molscal, a.phib_state, a.cbulk, cb);
      return;
    }
  }
  const long long i = (long long)blockIdx.x * kCB + threadIdx.x;
  if (i >= L.M) return;
  const int t = blockIdx.y;
  int x, y, z;
  site_coords(L, i, x, y, z);
  // halos from their sources; nothing behind a surface
  const int sx = remap(x, L.nx, L.b1[0], L.b2[0]);
  const int sy = L.grad >= 2 ? remap(y, L.ny, L.b1[1], L.b2[1]) : y;
  const int sz = L.grad >= 3 ? remap(z, L.nz, L.b1[2], L.b2[2]) : z;
  const long long s = sidx(L, sx, sy, sz);
  const bool surf_halo = !is_interior(L, sx, sy, sz);
  const long long ts = (long long)t * L.M + s, ti = (long long)t * L.M + i;
  double v = 0, dv = 0;
  if (a.frozen[t]) {
    if constexpr (BASE) v = a.fprof[ts];  // PutSides applies SetBoundaries to it as well
  } else if (!surf_halo) {
    const double g = a.swf[ts];
    double dir = 0;
    if constexpr (TAN) dir = a.vdir[ts];
    for (int m = 0; m < a.nm; m++) {
      if (!((a.uses[m] >> t) & 1u)) continue;
      const long long k = (long long)m * a.ns * L.M + ts;
      const bool mono = a.mode[m] == CLOSE_MONOMER;
      double p;
      if (!BASE || a.mode[m] == CLOSE_DONE) {
        p = a.phi_m[k];
      } else {
        const double pref = a.molscal[m * MS_COUNT + MS_PREF];
        p = mono ? pref * g
                 : phi_site((double)((const T*)a.acc)[k] + (a.two[m] ? (double)((const T*)a.acc2)[k] : 0.0), g, pref);
        if (s == i) a.phi_m[k] = p;
      }
      v += p;
      if constexpr (TAN) {
        const double da =
            mono ? 0.0 : (double)((const T*)a.dacc)[k] + (a.two[m] ? (double)((const T*)a.dacc2)[k] : 0.0);
        dv += tphi_site(mono, p, g, dir, da, a.dmol + m * 4);
      }
    }
  }
  if constexpr (BASE) a.phi[ti] = v;
  if constexpr (TAN) a.dphi[ti] = dv;
}

template <typename T>
void launch_phi_close(const DevLattice& L, const SysParams& sp, const PhiArgs& a, hipStream_t st) {
  const unsigned nb = grid1(L.M, kCB), ns = (unsigned)a.ns;
  if (a.base && a.tangent)
    k_phi_close<T, true, true><<<dim3(nb + 1, ns), kCB, 0, st>>>(L, sp, a);
  else if (a.base)
    k_phi_close<T, true, false><<<dim3(nb + 1, ns), kCB, 0, st>>>(L, sp, a);
  else
    k_phi_close<T, false, true><<<dim3(nb, ns), kCB, 0, st>>>(L, sp, a);
  SFX_HIP(hipGetLastError());
}
template void launch_phi_close<float>(const DevLattice&, const SysParams&, const PhiArgs&, hipStream_t);
template void launch_phi_close<double>(const DevLattice&, const SysParams&, const PhiArgs&, hipStream_t);

// ---------------------------------------------------------------------------
// NS: states whose averages are held in registers. All their loads are issued
// before the first is used, states past the last one repeating it: with a
// branch between states each waits for memory by itself (13 us for a product at
// 64 x 128). SFX_MAXS: any number of states one after the other, the averages
// read back from memory by the thread that wrote them.
// KIND: the lattice kind, ST_2D for all below three dimensions
template <int NS, int KIND, bool BASE, bool RES, bool TAN>
__global__ void __launch_bounds__(kCB) k_field_close(DevLattice L, SysParams sp, FieldArgs a) {
  const long long i = site_ordinal();
  if (i >= L.M) return;
  constexpr bool REG = NS < SFX_MAXS;
  constexpr int NR = REG ? NS : 1;
  int x, y, z;
  site_coords(L, i, x, y, z);
  const bool site = (RES || TAN) && a.itmask[i];
  const bool side = BASE ? has_side(L, x, y, z) : site;
  auto state = [&](int t) { return (long long)min(t, sp.ns - 1) * L.M; };
  double rr[NR], dr[NR], pt = 0, dpt = 0;
  if constexpr (REG) {
    double ph[NS], dp[NS];
#pragma unroll
    for (int t = 0; t < NS; t++) {
      ph[t] = BASE ? a.phi[state(t) + i] : 0.0;
      dp[t] = TAN ? a.dphi[state(t) + i] : 0.0;
      if constexpr (!BASE) rr[t] = a.rho[state(t) + i];
    }
    if constexpr (!BASE) pt = a.phitot[i];
    if constexpr (KIND >= ST_3D_SC) {  // sites without an average take one of the first layer and drop it
      const Near n = near_sites(L, side ? x : 1, side ? y : 1, side ? z : 1);
#pragma unroll
      for (int t = 0; t < NS; t++) {
        if constexpr (BASE) rr[t] = side_near<KIND>(n, a.phi + state(t));
        if constexpr (TAN) dr[t] = side_near<KIND>(n, a.dphi + state(t));
      }
    } else if (L.grad == 2) {
      const bool in = is_interior(L, x, y, 0);
      const Near2 n = near_sites2(L, in ? x : 1, in ? y : 1);
#pragma unroll
      for (int t = 0; t < NS; t++) {
        if constexpr (BASE) rr[t] = side_near2(L, n, a.phi + state(t));
        if constexpr (TAN) dr[t] = side_near2(L, n, a.dphi + state(t));
      }
      if (BASE && side && !in)  // a layer of a surface
#pragma unroll
        for (int t = 0; t < NS; t++) rr[t] = side_at2(L, a.phi + state(t), x, y);
    } else if (side) {
#pragma unroll
      for (int t = 0; t < NS; t++) {
        if constexpr (BASE) rr[t] = side_at1(L, a.phi + state(t), side_x1(L, x));
        if constexpr (TAN) dr[t] = side_at1(L, a.dphi + state(t), side_x1(L, x));
      }
    }
#pragma unroll
    for (int t = 0; t < NS; t++) {
      if (t >= sp.ns) break;
      if constexpr (BASE) {
        a.rho[(long long)t * L.M + i] = side ? rr[t] : 0.0;
        pt += ph[t];
      }
      if constexpr (TAN) dpt += dp[t];
    }
  } else {
    for (int t = 0; t < sp.ns; t++) {
      const long long k = (long long)t * L.M;
      if constexpr (BASE) {
        a.rho[k + i] = side ? side_at(L, a.phi + k, x, y, z) : 0.0;
        pt += a.phi[k + i];
      }
      if constexpr (TAN) {
        if (site) a.drho[k + i] = side_at(L, a.dphi + k, x, y, z);
        dpt += a.dphi[k + i];
      }
    }
    if constexpr (!BASE) pt = a.phitot[i];
  }
  if constexpr (BASE) a.phitot[i] = pt;
  auto rho = [&](int t) {
    if constexpr (REG)
      return rr[t];
    else
      return a.rho[(long long)t * L.M + i];
  };
  if constexpr (RES) {
    if (site)
      residual_site<NS>(sp, pt, a.cbulk, [&](int t) { return a.swf[(long long)t * L.M + i]; }, rho,
                        [&](int k, double v) { site_put(a.f, L.M, k, i, v); });
    else
      site_none(a.f, L.M, i);
  }
  if constexpr (TAN) {
    auto drho = [&](int t) {
      if constexpr (REG)
        return dr[t];
      else
        return a.drho[(long long)t * L.M + i];
    };
    if (site)
      jres_site<NS>(sp, pt, dpt, a.dmol, [&](int k) { return site_get(a.v, L.M, k, i); }, rho, drho,
                    [&](int k, double d) { site_put(a.jv, L.M, k, i, d); });
    else
      site_none(a.jv, L.M, i);
  }
}

template <int NS, int KIND>
static void field_close_k(const DevLattice& L, const SysParams& sp, const FieldArgs& a, hipStream_t st) {
  const unsigned nb = grid1(L.M, kCB);
  if (a.jv.p && a.base)
    k_field_close<NS, KIND, true, false, true><<<nb, kCB, 0, st>>>(L, sp, a);
  else if (a.jv.p)
    k_field_close<NS, KIND, false, false, true><<<nb, kCB, 0, st>>>(L, sp, a);
  else if (a.f.p)
    k_field_close<NS, KIND, true, true, false><<<nb, kCB, 0, st>>>(L, sp, a);
  else
    k_field_close<NS, KIND, true, false, false><<<nb, kCB, 0, st>>>(L, sp, a);
}
template <int NS>
static void field_close(const DevLattice& L, const SysParams& sp, const FieldArgs& a, hipStream_t st) {
  switch (L.kind) {
    case ST_3D_SC: field_close_k<NS, ST_3D_SC>(L, sp, a, st); break;
    case ST_3D_FCC: field_close_k<NS, ST_3D_FCC>(L, sp, a, st); break;
    case ST_3D_HEX: field_close_k<NS, ST_3D_HEX>(L, sp, a, st); break;
    default: field_close_k<NS, ST_2D>(L, sp, a, st); break;
  }
}

void launch_field_close(const DevLattice& L, const SysParams& sp, const FieldArgs& a, hipStream_t st) {
  if (sp.ns <= 2)
    field_close<2>(L, sp, a, st);
  else if (sp.ns <= 4)
    field_close<4>(L, sp, a, st);
  else
    field_close<SFX_MAXS>(L, sp, a, st);
  SFX_HIP(hipGetLastError());
}

}  // namespace sfx

// sfx_chain1d.hip -- a whole stretch of a chain's ranks on a 1-D lattice in
// one workgroup launch.
//
// A 1-D lattice has at most a few thousand sites, so one rank is a fraction
// of one workgroup's work and a launch per rank (SF_Copol1stO.cpp:1204-1232,
// one PropagateG per rank) is all launch overhead. Here one workgroup keeps
// the running rank in LDS (two ping-pong buffers indexed by layer, halos
// never stored: the stencil reads the remapped interior layer or 0 across a
// surface) and advances it through every step of the list with one barrier
// per rank; a step stores its rank to HBM when the backward pass needs it
// (`out`) and composes acc += G * pair (ConnectG) when it has a partner. The
// per-site arithmetic is that of k_prop, so the results are the same bits.
#include <atomic>

#include "sfx_chain1d.h"
#include "sfx_chain1w.h"
#include "sfx_scf.h"

namespace sfx {

constexpr int kC1Threads = 512;

__global__ void __launch_bounds__(kC1Threads) k_chain1d(DevLattice L, const double* __restrict__ in0,
                                                       const Chain1Step* __restrict__ steps, int n,
                                                       double* __restrict__ last) {
  extern __shared__ double lds[];
  const int nx = L.nx;
  double* cur = lds;
  double* nxt = lds + (nx + 2);
  for (int x = 1 + (int)threadIdx.x; x <= nx; x += kC1Threads) cur[x] = in0[sidx(L, x, 0, 0)];
  __syncthreads();
  for (int k = 0; k < n; k++) {
    const Chain1Step s = steps[k];
    for (int x = 1 + (int)threadIdx.x; x <= nx; x += kC1Threads) {
      const long long r = sidx(L, x, 0, 0);
      const double v = s.g[r] * stencil<double, ST_1D>(L, cur, x, 0, 0);
      nxt[x] = v;
      if (s.out) s.out[r] = v;
      if (s.acc) {
        const double cfac = 1.0;
        s.acc[r] = s.acc[r] + (double)(v * s.pair[r] * cfac);
      }
    }
    __syncthreads();
    double* t = cur;
    cur = nxt;
    nxt = t;
  }
  if (last)
    for (int x = 1 + (int)threadIdx.x; x <= nx; x += kC1Threads) last[sidx(L, x, 0, 0)] = cur[x];
}

bool chain1d_ok(const DevLattice& L) { return L.grad == 1 && L.order == 1 && L.nx >= 1 && L.nx <= kChain1MaxSites; }

void launch_chain1d(const DevLattice& L, const double* in0, const Chain1Step* steps, int n, double* last,
                    hipStream_t st) {
  const size_t lds = 2 * (size_t)(L.nx + 2) * sizeof(double);
  k_chain1d<<<1, kC1Threads, lds, st>>>(L, in0, steps, n, last);
}

// ---------------------------------------------------------------------------
// A whole evaluation of a 1-D system in one workgroup. It takes the place of
// the 22 launches of a residual (2-22 us each, most of them at the launch
// floor) and of the 150 to 300 of a product. 100 layers, A_100: 20 us of
// dependent steps (chain 9 us, molecule constants 4 us, the residual's logs 3
// us, the rest latencies) instead of 106 us of kernels, 136 -> 38 us a call; a
// product of 237 layers and 151 segments about 40 us instead of 600, 720 -> 58
// us a call. Four layers a lane (897 to 1024 layers) with tangents spill 107
// registers (flat; 164 curved), two 6 (15): a product of 1000 layers takes 160
// us all the same, 756 by launches.
// Larger lattices (1025 to 4000 layers), lattices of at most kChain1Halo layers
// and systems whose arrays do not fit LDS keep the launches (k_chain1d).
// ---------------------------------------------------------------------------
constexpr int kScf1Waves = 8, kScf1Threads = 64 * kScf1Waves;
constexpr int kScf1Lds = 156 * 1024;  // of 160 KB, the static words beside it

// every lambda of the sweep is inlined: one that is not would put the whole ring
// of partner rows into memory
#define SFX_INLINE __attribute__((always_inline))

// words of LDS per layer of a system with ns states
__host__ __device__ constexpr int scf1_words(int ns, bool tangent) { return tangent ? 4 * ns + 6 : 2 * ns + 3; }

// The sweep of one molecule by the whole workgroup: forward ranks to the
// store, then the composing ranks (the rest of a palindrome's chain, or the
// backward chain) with the stored ranks, fetched kRing ranks ahead so that
// their latency hides behind the ranks in between. acc (and dacc) of the
// molecule's states are in LDS, zero before; fin (dfin) gets the end rank.
template <int K, bool CURVED, bool TAN>
__device__ void chain1_sweep(const DevLattice& L, const Chain1Mol& mo, RunWalk w, double* store, double* dstore,
                             int W, const double* lg, const double* lv, double* lacc, double* ldacc,
                             double* fin, double* dfin, double* xch) {
  constexpr int kBlock = K == 4 ? 4 : kChain1Halo;  // ranks between two looks at the runs
  constexpr int kRing = 2 * kBlock;
  Chain1<K, CURVED, TAN> c;
  c.init(L, W, xch);
  const long long M = L.M;
  const int N = mo.N, h = N / 2, nfwd = mo.kind == 2 ? h : N;
  w.start(mo.run0, 1);
  auto load = [&]() SFX_INLINE { c.load(lg + w.state() * W, lv + w.state() * W); };
  load();
  c.rank1();
  double *row = store, *drow = dstore;
  c.put(row, drow);
  auto store_one = [&]() SFX_INLINE {
    c.step();
    row += M;
    if constexpr (TAN) drow += M;
    c.put(row, drow);
  };
  int s = 2;
  while (s <= nfwd) {
    if (s + kBlock - 1 <= nfwd && w.same(kBlock)) {
      c.room(kBlock);
      if (c.active) {
#pragma unroll
        for (int d = 0; d < kBlock; d++) store_one();
      }
      s += kBlock;
    } else {
      if (w.next()) load();
      c.room(1);
      if (c.active) store_one();
      s++;
    }
  }
  double acc[K], dacc[TAN ? K : 1];
#pragma unroll
  for (int j = 0; j < K; j++) {
    acc[j] = 0.0;
    if constexpr (TAN) dacc[j] = 0.0;
  }
  int t, ncomp, slot;
  if (mo.kind == 2) {
    t = w.state();
    if (N & 1) {  // the middle rank meets itself
      if (w.next()) {
        t = w.state();
        load();
      }
      c.room(1);
      c.step();
#pragma unroll
      for (int j = 0; j < K; j++) {
        acc[j] = 0.5 * (c.G[j] * c.G[j]);
        if constexpr (TAN) dacc[j] = 0.5 * tan_compose(c.D[j], c.G[j], c.G[j], c.D[j]);
      }
    }
    ncomp = h;
    slot = h - 1;
  } else {
    // rank N of the backward chain is g, its partner the rank in registers
    w.start(mo.run0 + mo.nruns - 1, -1);
    t = w.state();
    double e[K], de[TAN ? K : 1];
#pragma unroll
    for (int j = 0; j < K; j++) {
      e[j] = c.G[j];
      if constexpr (TAN) de[j] = c.D[j];
    }
    load();
    c.rank1();
#pragma unroll
    for (int j = 0; j < K; j++) {
      acc[j] = c.G[j] * e[j];
      if constexpr (TAN) dacc[j] = tan_compose(c.D[j], e[j], c.G[j], de[j]);
    }
    ncomp = N - 1;
    slot = N - 2;
  }
  // the accumulators of state t go back to LDS, those of state `to` come
  auto flush = [&](int to) SFX_INLINE {
#pragma unroll
    for (int j = 0; j < K; j++) {
      lacc[t * W + c.to[j]] = acc[j];
      acc[j] = lacc[to * W + c.to[j]];
      if constexpr (TAN) {
        ldacc[t * W + c.to[j]] = dacc[j];
        dacc[j] = ldacc[to * W + c.to[j]];
      }
    }
    t = to;
  };
  double pr[kRing][K], dpr[TAN ? kRing : 1][TAN ? K : 1];
  // the next partner row, down to the first
  row = store + (long long)slot * M;
  drow = TAN ? dstore + (long long)slot * M : nullptr;
  auto fetch = [&](int d) SFX_INLINE {
    c.get(row, drow, pr[d], dpr[TAN ? d : 0]);
    const bool more = row != store;
    row -= more ? M : 0;
    if constexpr (TAN) drow -= more ? M : 0;
  };
  auto compose = [&](const double (&p)[K], const double (&dp)[TAN ? K : 1]) SFX_INLINE {
    c.step();
#pragma unroll
    for (int j = 0; j < K; j++) {
      acc[j] = fma(c.G[j], p[j], acc[j]);
      if constexpr (TAN) dacc[j] = dacc[j] + tan_compose(c.D[j], p[j], c.G[j], dp[j]);
    }
  };
  // `cnt` ranks with the rows b.. of the ring, one by one: near a change of
  // the state and at the chain's end
  auto slowly = [&](int b, int cnt) SFX_INLINE {
#pragma unroll 1
    for (int d = 0; d < cnt; d++) {
      if (w.next()) {
        load();
        if (w.state() != t) flush(w.state());
      }
      double p[K], dp[TAN ? K : 1];
#pragma unroll
      for (int j = 0; j < K; j++) {  // selected by value: an index would put the ring into memory
        p[j] = pr[b][j];
        if constexpr (TAN) dp[j] = dpr[b][j];
#pragma unroll
        for (int e = 1; e < kBlock; e++) {
          p[j] = d == e ? pr[b + e][j] : p[j];
          if constexpr (TAN) dp[j] = d == e ? dpr[b + e][j] : dp[j];
          asm volatile("" : "+v"(p[j]));  // keeps the selects apart: merged into an index, they too would
          if constexpr (TAN) asm volatile("" : "+v"(dp[j]));
        }
      }
      compose(p, dp);
    }
  };
#pragma unroll
  for (int d = 0; d < kRing; d++) fetch(d);
  int k = 0;
  while (k < ncomp) {
#pragma unroll
    for (int b = 0; b < kRing; b += kBlock) {
      const int cnt = min(kBlock, ncomp - k);
      if (cnt > 0) {
        c.room(kBlock);
        if (cnt == kBlock && w.same(kBlock)) {
          if (c.active) {
#pragma unroll
            for (int d = b; d < b + kBlock; d++) compose(pr[d], dpr[TAN ? d : 0]);
          }
        } else {
          slowly(b, cnt);
        }
        if (c.active && k + kRing < ncomp) {
#pragma unroll
          for (int d = 0; d < kBlock; d++) fetch(b + d);
        }
        k += kBlock;
      }
    }
  }
  flush(t);
#pragma unroll
  for (int j = 0; j < K; j++) {
    fin[c.to[j]] = c.G[j];
    if constexpr (TAN) dfin[c.to[j]] = c.D[j];
  }
}

// sums over the interior layers of val(x) and, with TAN, dval(x), added up as
// the per-launch kernels do (a workgroup of four waves per 256 layers, then a
// wave over the workgroups); every thread gets them. wsum: 32 words, no one
// reads them before the first barrier here
template <bool TAN, class Val, class Dval>
__device__ double2 scf1_layer_sums(int n, Val&& val, Dval&& dval, double* wsum) {
  const int lane = (int)threadIdx.x & 63;
  for (int w = (int)threadIdx.x >> 6; w < 16; w += kScf1Waves) {
    const int x = 1 + w * 64 + lane;
    double v = 0.0, d = 0.0;
    if (w * 64 < n) {  // wave-uniform
      if (x <= n) {
        v = val(x);
        if constexpr (TAN) d = dval(x);
      }
#pragma unroll 1
      for (int o = 32; o > 0; o >>= 1) {
        v += __shfl_xor(v, o, 64);
        if constexpr (TAN) d += __shfl_xor(d, o, 64);
      }
    }
    if (lane == 0) {
      wsum[w] = v;
      if constexpr (TAN) wsum[16 + w] = d;
    }
  }
  __syncthreads();
  double s = 0.0, d = 0.0;
  if (lane < 4 && lane * 256 < n)
    for (int i = 0; i < 4; i++) {
      s += wsum[lane * 4 + i];
      if constexpr (TAN) d += wsum[16 + lane * 4 + i];
    }
  // the other lanes hold 0: a wave's butterfly leaves (0 + 2) + (1 + 3) of the first four
#pragma unroll
  for (int o = 2; o > 0; o >>= 1) {
    s += __shfl_xor(s, o, 64);
    if constexpr (TAN) d += __shfl_xor(d, o, 64);
  }
  s = __shfl(s, 0, 64);
  if constexpr (TAN) d = __shfl(d, 0, 64);
  __syncthreads();
  return make_double2(s, d);
}

// The residual (u -> SWF -> propagators -> phi -> f), or with TAN the product
// J v (A.base: with phi and the contact averages on the way; otherwise at those
// of the last evaluation), of a 1-D first-order system in FP64: the launches of a
// residual or a product in one workgroup; a residual's bits are the launches'.
// SWF, accumulators and profiles are in LDS, indexed by layer with W words per
// state; every wave sweeps its layers of the chains.
template <int K, bool CURVED, bool TAN>
__global__ void __launch_bounds__(kScf1Threads) k_scf1d(DevLattice L, Scf1Args A) {
  extern __shared__ double lds[];
  __shared__ double wsum[32], cb[SFX_MAXS], ms[SFX_MAXM * MS_COUNT], dm[SFX_MAXM * 4];
  const SysParams& sp = A.sp;
  const int ns = sp.ns, n = L.nx, M = n + 2, W = M, tid = (int)threadIdx.x;
  const bool base = !TAN || A.base;
  double* lg = lds;
  double* lacc = lg + ns * W;  // accumulators, then phi
  double* fin = lacc + ns * W;
  double* xch = fin + W;  // exchange buffers of the chain: 2 ranks (4 with tangents)
  double* lv = TAN ? xch + 4 * W : lds;
  double* ldacc = TAN ? lv + ns * W : lds;  // accumulators, then dphi
  double* dfin = TAN ? ldacc + ns * W : lds;

  for (int i = tid; i < scf1_words(ns, TAN) * W; i += kScf1Threads) lds[i] = 0.0;
  RunWalk walk;
  walk.init(A.runs, A.nruns);
  if (!base && tid < sp.nm * MS_COUNT) ms[tid] = tid % MS_COUNT == MS_REF || tid % MS_COUNT == MS_POW ? 0.0 : A.molscal[tid];
  __syncthreads();
  if (A.u)
    for (int q = tid; q < sp.n_itvar * M; q += kScf1Threads) A.u[q] = site_get(A.x, M, q / M, q % M);
  // SWF (k_swf), a thread per state and layer
  for (int q = tid; q < ns * M; q += kScf1Threads) {
    const int t = q / M, i = q - t * M;
    const int s = remap(i, n, L.b1[0], L.b2[0]);
    const int iv = sp.st_itvar[t];
    const double g = (iv >= 0 && A.itmask[s]) ? exp(-site_get(A.x, M, iv, s)) : 0.0;
    if (i >= 1 && i <= n) {
      lg[t * W + i] = g;
      if constexpr (TAN) lv[t * W + i] = iv >= 0 ? site_get(A.v, M, iv, i) : 0.0;
    }
    if (base) {
      A.swf[(long long)t * M + i] = g;
      A.swf32[(long long)t * M + i] = (float)g;
    }
  }
  __syncthreads();

#pragma unroll 1
  for (int k = 0; k < sp.nm; k++) {
    const Chain1Mol& mo = A.mols[k];  // non-solvent molecules first
    const MolParams mp{mo.index, mo.N, mo.freedom, mo.kind, mo.phib, mo.theta};
    double* mscal = ms + mo.index * MS_COUNT;
    double* phi_m = A.phi_m + (long long)mo.index * ns * M;
    double* dphi_m = TAN ? A.dphi_m + (long long)mo.index * ns * M : nullptr;
    const int t0 = __ffs(mo.uses) - 1;  // a monomer's state
    if (mo.kind != 0) {
      if (mo.uses & A.shared) {  // another molecule's phi of these states is there
        for (int t = 0; t < ns; t++)
          if ((mo.uses >> t) & 1u)
            for (int i = tid; i < W; i += kScf1Threads) {
              lacc[t * W + i] = 0.0;
              if constexpr (TAN) ldacc[t * W + i] = 0.0;
            }
        __syncthreads();
      }
      chain1_sweep<K, CURVED, TAN>(L, mo, walk, A.store, A.dstore, W, lg, lv, lacc,
                                   ldacc, fin, dfin, xch);
      __syncthreads();
    }
    const double* end = mo.kind == 0 ? lg + t0 * W : fin;
    const double2 sums = scf1_layer_sums<TAN>(
        n, [&](int x) { return end[x] * lngn_weight1(L, x); },
        [&](int x) {
          const double d = mo.kind == 0 ? -lv[t0 * W + x] * lg[t0 * W + x] : dfin[x];
          return d * lngn_weight1(L, x);
        },
        wsum);
    if (base) {
      if (tid == 0) {
        mscal[MS_REF] = mscal[MS_POW] = 0.0;
        mol_scalars(mp, sums.x, 0.0, 0.0, 0, sp.nm, [&](int m) { return ms[m * MS_COUNT + MS_PHIB]; }, mscal);
      }
      __syncthreads();
      const double pref = mscal[MS_PREF];
      for (int x = 1 + tid; x <= n; x += kScf1Threads)
        for (int t = 0; t < ns; t++)
          if ((mo.uses >> t) & 1u) {
            const double g = lg[t * W + x];
            const double ph = mo.kind == 0 ? pref * g : phi_site(lacc[t * W + x], g, pref);
            lacc[t * W + x] = ph;
            phi_m[(long long)t * M + x] = ph;
          }
      if (mo.freedom == SFX_RANGE_RESTRICTED) {
        __syncthreads();
        const double2 s = scf1_layer_sums<false>(
            n,
            [&](int x) {
              double v = 0;
              if (x >= mo.lo && x <= mo.hi)
                for (int t = 0; t < ns; t++)
                  if (mo.uses >> t & 1u) v += lacc[t * W + x];
              return v;
            },
            [](int) { return 0.0; }, wsum);
        if (tid == 0) range_scalars(s.x, mo.phi_range, mo.N, mscal);
        __syncthreads();
        const double C = mscal[MS_RANGE_C];
        for (int x = 1 + tid; x <= n; x += kScf1Threads)
          for (int t = 0; t < ns; t++)
            if (mo.uses >> t & 1u) {
              lacc[t * W + x] *= C;
              phi_m[(long long)t * M + x] = lacc[t * W + x];
            }
      }
    } else {
      for (int x = 1 + tid; x <= n; x += kScf1Threads)
        for (int t = 0; t < ns; t++)
          if ((mo.uses >> t) & 1u) lacc[t * W + x] = phi_m[(long long)t * M + x];
    }
    if constexpr (TAN) {
      if (tid == 0)
        tmol_scalars(mp, true, sums.x, sums.y, mscal, sp.nm, [&](int m) { return dm[m * 4 + 2]; }, dm + mo.index * 4);
      __syncthreads();
      for (int x = 1 + tid; x <= n; x += kScf1Threads)
        for (int t = 0; t < ns; t++)
          if ((mo.uses >> t) & 1u) {
            const double d = tphi_site(mo.kind == 0, lacc[t * W + x], lg[t * W + x], lv[t * W + x],
                                       ldacc[t * W + x], dm + mo.index * 4);
            ldacc[t * W + x] = d;
            dphi_m[(long long)t * M + x] = d;
          }
    }
    __syncthreads();
  }

  // state totals (k_phi_close): a state of one molecule has its
  // phi in LDS; one of several is summed over the phi_m this thread wrote
  for (int x = 1 + tid; x <= n; x += kScf1Threads)
    for (int t = 0; t < ns; t++) {
      if (sp.frozen[t]) {
        lacc[t * W + x] = A.fprof[(long long)t * M + x];
      } else if ((A.shared >> t) & 1u) {
        double v = 0, d = 0;
        for (int m = 0; m < sp.nm; m++)
          if (sp.mol_frac[m * SFX_MAXS + t] > 0) {
            v += A.phi_m[((long long)m * ns + t) * M + x];
            if constexpr (TAN) d += A.dphi_m[((long long)m * ns + t) * M + x];
          }
        lacc[t * W + x] = v;
        if constexpr (TAN) ldacc[t * W + x] = d;
      }
    }
  if (base && tid >= kScf1Threads - 64) bulk_fractions_wave(sp, ms, A.phib_state, A.cbulk, cb);
  __syncthreads();
  // halo layers from their sources
  if (tid < 2 * ns) {
    const int t = tid >> 1, i = tid & 1 ? n + 1 : 0;
    const int s = remap(i, n, L.b1[0], L.b2[0]);
    const bool surf_halo = s < 1 || s > n;
    lacc[t * W + i] = sp.frozen[t] ? A.fprof[(long long)t * M + s] : (surf_halo ? 0.0 : lacc[t * W + s]);
    if constexpr (TAN) ldacc[t * W + i] = (sp.frozen[t] || surf_halo) ? 0.0 : ldacc[t * W + s];
  }
  if (base && tid < sp.nm * MS_COUNT) A.molscal[tid] = ms[tid];
  __syncthreads();
  // contact averages and the residual or its linearisation
  for (int i = tid; i < M; i += kScf1Threads) {
    double tot = 0, dtot = 0;
    for (int t = 0; t < ns; t++) {
      tot += lacc[t * W + i];
      if constexpr (TAN) dtot += ldacc[t * W + i];
    }
    const SiteOut& out = TAN ? A.jv : A.f;
    const bool side = (i > 0 || L.surf1[0]) && (i <= n || L.surf2[0]);  // not the other halos
    if (base) {
      A.phitot[i] = tot;
      for (int t = 0; t < ns; t++) {
        A.phi[(long long)t * M + i] = lacc[t * W + i];
        A.rho[(long long)t * M + i] = side ? side_at1(L, lacc + t * W, i) : 0.0;
      }
    }
    if (!out.p) continue;
    if (!A.itmask[i]) {
      site_none(out, M, i);
      continue;
    }
    auto rho = [&](int t) { return base ? side_at1(L, lacc + t * W, i) : A.rho[(long long)t * M + i]; };
    if constexpr (TAN) {
      jres_site(sp, tot, dtot, dm, [&](int k) { return site_get(A.v, M, k, i); }, rho,
                [&](int t) { return side_at1(L, ldacc + t * W, i); },
                [&](int k, double d) { site_put(out, M, k, i, d); });
    } else {
      residual_site(sp, tot, cb, [&](int t) { return lg[t * W + i]; }, rho,
                    [&](int k, double v) { site_put(out, M, k, i, v); });
    }
  }
}

// slots per lane: the fewest that hold the lattice. One slot per lane is the
// shortest chain of dependent instructions per rank
static int scf1_k(int n) {
  return n <= kScf1Waves * chain1_owned(1) ? 1 : n <= kScf1Waves * chain1_owned(2) ? 2 : 4;
}
static size_t scf1_lds(int n, int ns, bool tangent) {
  return (size_t)scf1_words(ns, tangent) * (n + 2) * sizeof(double);
}

bool scf1d_ok(const DevLattice& L, int ns, bool tangent) {
  return L.grad == 1 && L.order == 1 && L.nx > kChain1Halo && L.nx <= 1024 &&
         scf1_lds(L.nx, ns, tangent) <= kScf1Lds;
}

template <int K, bool CURVED, bool TAN>
static void scf1_launch(const DevLattice& L, const Scf1Args& a, hipStream_t st) {
  const size_t lds = scf1_lds(L.nx, a.sp.ns, TAN);
  if (lds > 64 * 1024) {  // dynamic LDS beyond the default needs the attribute, once per device
    static std::atomic<unsigned> set{0};
    int dev = 0;
    SFX_HIP(hipGetDevice(&dev));
    const unsigned bit = 1u << (dev & 31);
    if (!(set.load() & bit)) {
      SFX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_scf1d<K, CURVED, TAN>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, kScf1Lds));
      set.fetch_or(bit);
    }
  }
  k_scf1d<K, CURVED, TAN><<<1, kScf1Threads, lds, st>>>(L, a);
}

template <bool TAN>
static void scf1_launch_k(const DevLattice& L, const Scf1Args& a, hipStream_t st) {
#define SCF1(K)                                      \
  if (L.curved) scf1_launch<K, true, TAN>(L, a, st); \
  else scf1_launch<K, false, TAN>(L, a, st)
  switch (scf1_k(L.nx)) {
    case 1: SCF1(1); break;
    case 2: SCF1(2); break;
    default: SCF1(4); break;
  }
#undef SCF1
  SFX_HIP(hipGetLastError());
}

void launch_scf1d(const DevLattice& L, const Scf1Args& a, bool tangent, hipStream_t st) {
  SFX_REQUIRE(scf1d_ok(L, a.sp.ns, tangent), SFX_E_INVALID, "1-D system too large for one workgroup");
  if (tangent) scf1_launch_k<true>(L, a, st);
  else scf1_launch_k<false>(L, a, st);
}

}  // namespace sfx

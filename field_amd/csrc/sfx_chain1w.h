// sfx_chain1w.h -- the running rank of a chain on a 1-D lattice in the
// registers of one workgroup (device code; sfx_chain1d.hip, sfx_batch.hip).
#pragma once

#include "sfx_chain1d.h"
#include "sfx_scf.h"

namespace sfx {

// A wave holds 64 K consecutive layers, K per lane: the layers it owns and, at
// either end, kChain1Halo layers of its neighbours. Without anything from
// outside it advances kChain1Halo ranks, its valid part shrinking by one layer
// at either end per rank; then the workgroup exchanges a rank through LDS with
// one barrier. Layers behind a bound are images of interior layers (their g
// and, on curved lattices, their weights mirrored with them), behind a surface
// 0. What bounds it: the operations of a rank one after the other. Two wave
// shifts and five FP64 operations take 54 cycles, the rank's store 16, an eighth
// of an exchange 30 (measured on 100 layers, one layer per lane); a rank kept in
// LDS, with a barrier each (k_chain1d), took 430 ns, 900 cycles. Sixteen layers
// of halo would halve the exchange's share but lose a third of a wave's layers.
constexpr int kChain1Halo = 8;
__host__ __device__ constexpr int chain1_owned(int K) { return 64 * K - 2 * kChain1Halo; }

// the value of the lane below / above (0 beyond the wave's ends), on the
// vector unit: a double moves as two words
__device__ __forceinline__ double from_below(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x138, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x138, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double from_above(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x130, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x130, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// Every thread of the workgroup calls every member; xch: LDS for 2 ranks (4
// with tangents) of W words, zero at index 0. BATCH: the batched problems' own
// step (surface below, mirror1 above by value, its operations in their order:
// their DIIS iterates depend on the last bit of a residual).
template <int K, bool CURVED, bool TAN, bool BATCH = false>
struct Chain1 {
  double G[K], g[K], D[TAN ? K : 1], v[TAN ? K : 1];
  double lm[CURVED ? K : 1], lp[CURVED ? K : 1];
  double l1;
  int x[K];      // the interior layer of slot j, or the one it is the image of (0: nothing)
  int to[K];     // where slot j's value goes: its layer if it is owned, else n + 1, which nobody reads
  bool last[BATCH ? K : 1];  // layer n
  bool active;   // this wave owns any; the others only keep the barriers
  double* xch;
  int W, since, buf;

  __device__ __forceinline__ void init(const DevLattice& L, int W_, double* xch_) {
    W = W_;
    xch = xch_;
    l1 = L.l1;
    since = buf = 0;
    const int n = L.nx, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    active = wave * chain1_owned(K) < n;
#pragma unroll
    for (int j = 0; j < K; j++) {
      const int i = lane * K + j;
      int c = wave * chain1_owned(K) + 1 - kChain1Halo + i;
      to[j] = i >= kChain1Halo && i < 64 * K - kChain1Halo && c <= n ? c : n + 1;
      bool image = false;
      if (c < 1) {
        image = !L.periodic[0];
        c = L.surf1[0] ? 0 : (L.periodic[0] ? c + n : (L.mirror2_1[0] ? 2 - c : 1 - c));
      } else if (c > n) {
        image = !L.periodic[0];
        c = L.surf2[0] ? 0 : (L.periodic[0] ? c - n : (L.mirror2_2[0] ? 2 * n - c : 2 * n + 1 - c));
      }
      if constexpr (BATCH) {
        last[j] = !image && c == n;
        if (image) c = 0;
      }
      x[j] = c < 1 || c > n ? 0 : c;  // farther out: never reaches an owned layer
      if constexpr (CURVED) {
        lm[j] = image ? L.lp[x[j]] : L.lm[x[j]];
        lp[j] = image ? L.lm[x[j]] : L.lp[x[j]];
      }
    }
  }
  // SWF (and direction) of a state, arrays indexed by layer with 0 at index 0
  __device__ __forceinline__ void load(const double* lg, const double* lv) {
#pragma unroll
    for (int j = 0; j < K; j++) {
      g[j] = lg[x[j]];
      if constexpr (TAN) v[j] = lv[x[j]];
    }
  }
  __device__ __forceinline__ void rank1() {
    since = 0;
#pragma unroll
    for (int j = 0; j < K; j++) {
      G[j] = g[j];
      if constexpr (TAN) D[j] = -v[j] * g[j];
    }
  }
  __device__ __forceinline__ void average(const double (&P)[K], double (&A)[K]) const {
    double a = from_below(P[K - 1]);
    const double above = from_above(P[0]);
#pragma unroll
    for (int j = 0; j < K; j++) {
      const double c = j + 1 < K ? P[j + 1 < K ? j + 1 : j] : above;
      if constexpr (BATCH) A[j] = fma(l1, fma(-2.0, P[j], a) + (last[j] ? P[j] : c), P[j]);
      else if constexpr (CURVED) A[j] = step1_curved(lm[j], lp[j], a, P[j], c);
      else A[j] = step1_flat(l1, a, P[j], c);
      a = P[j];
    }
  }
  __device__ __forceinline__ void exchange() {
    double* const b = xch + buf * (TAN ? 2 : 1) * W;
    if (active) {
#pragma unroll
      for (int j = 0; j < K; j++) {
        b[to[j]] = G[j];
        if constexpr (TAN) (b + W)[to[j]] = D[j];
      }
    }
    __syncthreads();
    if (active) {
#pragma unroll
      for (int j = 0; j < K; j++) {
        G[j] = b[x[j]];
        if constexpr (TAN) D[j] = (b + W)[x[j]];
      }
    }
    buf ^= 1;  // the other buffer next: a slower wave may still read this one
    since = 0;
  }
  // room for `ranks` (at most kChain1Halo) ranks without an exchange
  __device__ __forceinline__ void room(int ranks) {
    if (since + ranks > kChain1Halo) exchange();
    since += ranks;
  }
  // the next rank, after room()
  __device__ __forceinline__ void step() {
    double A[K];
    average(G, A);
    if constexpr (TAN) {
      double dA[K];
      average(D, dA);
#pragma unroll
      for (int j = 0; j < K; j++) D[j] = g[j] * tan_step(dA[j], v[j], A[j]);
    }
#pragma unroll
    for (int j = 0; j < K; j++) G[j] = g[j] * A[j];
  }
  // the owned layers to a rank's row in the store, and a partner's from it. No
  // lane is masked off (that costs more than the rank's arithmetic): lanes
  // without a layer all use the row's last word, the upper halo, so no kernel
  // may read that word of a 1-D store
  static __device__ __forceinline__ double& at(double* row, int i) {
    return *(double*)((char*)row + (unsigned)(i * 8));
  }
  __device__ __forceinline__ void put(double* row, double* drow) const {
#pragma unroll
    for (int j = 0; j < K; j++) {
      at(row, to[j]) = G[j];
      if constexpr (TAN) at(drow, to[j]) = D[j];
    }
  }
  __device__ __forceinline__ void get(double* row, double* drow, double (&p)[K], double (&dp)[TAN ? K : 1]) const {
#pragma unroll
    for (int j = 0; j < K; j++) {
      p[j] = at(row, to[j]);
      if constexpr (TAN) dp[j] = at(drow, to[j]);
    }
  }
};

// the state runs of a chain, forwards or backwards from either end; the first
// 64 runs of the system are in registers, one per lane
struct RunWalk {
  const Chain1Run* run;
  int state_of, count_of;  // this lane's run
  int i, step, left, st;
  __device__ __forceinline__ void init(const Chain1Run* r, int nruns) {
    run = r;
    const int lane = (int)threadIdx.x & 63;
    state_of = count_of = 0;
    if (lane < nruns) {
      state_of = r[lane].state;
      count_of = r[lane].count;
    }
  }
  __device__ __forceinline__ void set() {
    if (i < 64) {
      left = __builtin_amdgcn_readlane(count_of, i);
      st = __builtin_amdgcn_readlane(state_of, i);
    } else {
      left = __builtin_amdgcn_readfirstlane(run[i].count);
      st = __builtin_amdgcn_readfirstlane(run[i].state);
    }
  }
  __device__ __forceinline__ void start(int first, int step_) {
    i = first;
    step = step_;
    set();
  }
  __device__ __forceinline__ int state() const { return st; }
  // to the next rank; true when its state may be another one
  __device__ __forceinline__ bool next() {
    if (--left > 0) return false;
    i += step;
    set();
    return true;
  }
  // whether the next `ranks` ranks have the state of the current one; passes them
  __device__ __forceinline__ bool same(int ranks) {
    if (left <= ranks) return false;
    left -= ranks;
    return true;
  }
};

}  // namespace sfx

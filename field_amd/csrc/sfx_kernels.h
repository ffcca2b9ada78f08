// sfx_kernels.h -- launch wrappers and kernel parameter blocks.
#pragma once

#include "sfx_internal.h"

#define SFX_MAXS 8  // segment states per system
#define SFX_MAXM 8  // molecules per system

namespace sfx {

// per-molecule device scalars
enum { MS_LNGN = 0, MS_LNC, MS_PHIB, MS_PREF, MS_REF, MS_RANGE_C, MS_POW, MS_COUNT = 8 };

// FP32 per-rank log-scaling context of one sweep. Step k writes max|G| of its
// output into maxv[k] and the cumulative log scale into lnv[k]; its output is
// multiplied by 1/maxv[k-1]. Composition multiplies by
// exp(lnv[k] + lnpair[pair] - *ref). maxv == nullptr disables scaling.
// The maximum of a step is spread over kMaxSlots words (workgroup b writes
// word b mod kMaxSlots), kSlotStride words apart: atomics on one line
// serialise, and a per-rank launch on a large lattice has thousands of
// workgroups. A reader reduces the words with one wave load, so every line more
// costs it too: a second-order product at 128^3 took 32.9 ms with a line per
// word, 32.2 ms with four words a line, 35.2 ms with all in two lines. A step
// occupies kStepWords words.
constexpr int kMaxSlots = 64;
constexpr int kSlotStride = 8;  // 32 bytes
constexpr int kStepWords = kMaxSlots * kSlotStride;

__device__ __forceinline__ void put_step_max(unsigned* maxv, int step, float m) {
  atomicMax(maxv + (long long)step * kStepWords + (blockIdx.x & (kMaxSlots - 1)) * kSlotStride,
            __float_as_uint(m));
}

// the maxima of two steps (a second pointer may be null: its value is 0),
// read once per workgroup by its first wave (one slot line per lane) and shared
// through LDS; every thread of the workgroup must call it
__device__ __forceinline__ void block_step_max2(const unsigned* maxa, int sa, const unsigned* maxb, int sb,
                                                float& ma, float& mb) {
  __shared__ float sh[2];
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    float a = __uint_as_float(maxa[(long long)sa * kStepWords + lane * kSlotStride]);
    float b = maxb ? __uint_as_float(maxb[(long long)sb * kStepWords + lane * kSlotStride]) : 0.f;
    for (int o = 32; o > 0; o >>= 1) {
      a = fmaxf(a, __shfl_xor(a, o, 64));
      b = fmaxf(b, __shfl_xor(b, o, 64));
    }
    if (lane == 0) {
      sh[0] = a;
      sh[1] = b;
    }
  }
  __syncthreads();
  ma = sh[0];
  mb = sh[1];
}

// A launch of several ranks divides by the lattice maximum of g alone, so its
// ranks decay wherever the chain's weight is far from that maximum (an isolated
// deep site, a block entering another's region, strong noise). Its ranks carry a
// factor kBlockScale = 2^32 (their values and maxima; lnv is the log without it),
// and where a launch's last rank has fallen below kLowMax = 2^-24 of its input (17
// kT) the evaluation is repeated rank by rank. The accumulators carry 2^MS_POW,
// which puts the ranks that the reference log is taken from at 2^kAccPower. So
// every rank, composed product and accumulator has at least the range above FP32's
// smallest numbers that the per-rank kernels leave it, whose ranks are at most g's
// maximum (up to exp(5.5)). With a maximum of 1 and no check, transposed products
// lost digits from a loss of 2^-60 on, sums of 2^-127 became log(0), and a profile
// fixed by its amount in a box far from the chain's weight came out 0. Powers of
// two round nothing: a field without such decays gives the bits it gave without.
constexpr int kBlockPower = 32, kAccPower = 32;
constexpr float kBlockScale = 0x1p32f, kBlockDown = 0x1p-32f;
constexpr float kLowMax = 0x1p-24f;
// a launch's input of maximum m (without kBlockScale) has decayed too far; or, if it
// is a first rank, which does not carry the factor yet, kBlockScale / m may be no
// number (a field of 62 kT everywhere)
__host__ __device__ constexpr bool low_input(float m, bool carried) { return !(m >= (carried ? kLowMax : 0x1p-90f)); }

struct RankScale {
  unsigned* maxv;
  double* lnv;
  const double* lnpair;
  const double* ref;
  int step;
  int pair;
  const unsigned* pmaxv = nullptr;  // step maxima of the partner chain (second order recovers its rank)
  // beside blocked launches: rank step - 1 carries kBlockScale; a composition in
  // their accumulators (MS_POW), of `carry` ranks that carry it
  bool prev_blocked = false;
  const double* pow = nullptr;
  int carry = 0;
};

#ifdef __HIPCC__
__device__ __forceinline__ double connect_factor(const RankScale& sc, double half) {
  const double c = half * exp(sc.lnv[sc.step] + sc.lnpair[sc.pair] - *sc.ref);
  return sc.pow ? ldexp(c, (int)*sc.pow - kBlockPower * sc.carry) : c;
}
#endif

struct MolParams {
  int index, N, freedom, kind;  // kind: 0 monomer, 1 full sweep, 2 half-stored (palindrome), 3 second order
  double phib, theta;
};

struct SysParams {
  int ns, nm, n_itvar, melt;
  double chi[SFX_MAXS * SFX_MAXS];
  int frozen[SFX_MAXS];
  int st_itvar[SFX_MAXS];
  int itvar_rep[SFX_MAXS];
  double melt_phib[SFX_MAXS];
  double mol_frac[SFX_MAXM * SFX_MAXS];
  double mol_N[SFX_MAXM];
  double mol_ref[SFX_MAXM];
};

// A vector over the iteration variables, read or written by the kernels in the
// layout it has: p[k * M + i] for variable k of site i, or, where order is
// given, the variables of a site together in the order of the iteration sites
// (sfx_residual's layout of the SF form). Sites off the iteration read 0.
struct SiteVec {
  const double* p;
  const int* order;            // site -> its ordinal, -1 off the iteration
  const unsigned char* mask;
  int nv;
};
struct SiteOut {
  double* p;  // may be null
  const int* order;
  int nv;
};
#ifdef __HIPCC__
__device__ __forceinline__ double site_get(const SiteVec& v, long long M, int k, long long i) {
  if (v.order) {
    const int o = v.order[i];
    return o >= 0 ? v.p[(long long)o * v.nv + k] : 0.0;
  }
  return v.mask[i] ? v.p[(long long)k * M + i] : 0.0;
}
__device__ __forceinline__ void site_put(const SiteOut& f, long long M, int k, long long i, double value) {
  f.p[f.order ? (long long)f.order[i] * f.nv + k : (long long)k * M + i] = value;
}
// a site off the iteration: 0, where the layout has a place for it
__device__ __forceinline__ void site_none(const SiteOut& f, long long M, long long i) {
  if (!f.order)
    for (int k = 0; k < f.nv; k++) f.p[(long long)k * M + i] = 0.0;
}
#endif

// device arrays of 4-byte words cleared by one launch
struct ZeroList {
  static constexpr int max = 24;
  void* p[max];
  long long words[max];
  int n = 0;
};
void launch_zero_list(const ZeroList& z, hipStream_t st);
// adds an array, launching the list first when it is full
void zero_list_add(ZeroList& z, void* p, long long words, hipStream_t st);

template <typename T, typename A>
void launch_prop(const DevLattice& L, const T* Gin, const T* g, T* Gout, const T* Gpair, A* acc,
                 const RankScale& sc, hipStream_t st);
template <typename T>
void launch_init_rank(const DevLattice& L, const T* g, T* out, const RankScale& sc, hipStream_t st);
// rank 1 of two chains (the forward and backward ends of a middle-out sweep) in one launch
template <typename T>
struct InitRank {
  const T* g;
  T* out;
  RankScale sc;
};
template <typename T>
void launch_init_rank2(const DevLattice& L, const InitRank<T>& c0, const InitRank<T>& c1, hipStream_t st);
template <typename T, typename A>
void launch_connect(const DevLattice& L, const T* a, const T* b, A* acc, const RankScale& sc, double half,
                    hipStream_t st);
template <typename T>
void launch_copy_interior(const DevLattice& L, const T* a, T* b, hipStream_t st);
template <typename T>
int launch_wsum(const DevLattice& L, const T* G, double* partial, hipStream_t st);
// phi_m = pref (acc + acc2) / g; acc2 (the backward chain's accumulator of a
// middle-out sweep) may be null
template <typename A>
void launch_mol_phi(const DevLattice& L, const A* acc, const double* g, const double* scal, int monomer,
                    double* phi_m, hipStream_t st, const A* acc2 = nullptr);
// phi_m of every state set in `uses` in one launch (state-major arrays from the given bases)
template <typename A>
void launch_mol_phi_states(const DevLattice& L, unsigned uses, int ns, const A* acc, const A* acc2, const double* g,
                           const double* scal, double* phi_m, hipStream_t st);
// scal[MS_REF], scal[MS_POW] = the reference log of a blocked sweep's compositions
// and their accumulators' power of two, from the logs and maxima of the ranks that
// the chains' first halves end with (lnb null: of one)
void launch_set_ref_block(double* scal, const unsigned* maxa, const double* lna, int ia, const unsigned* maxb,
                          const double* lnb, int ib, hipStream_t st);
// The SWF of every state, and what else a sweep needs beside it: x's copy in
// the internal layout, arrays to be cleared, a product's direction per state
struct SwfArgs {
  SiteVec x;
  double* u;  // may be null
  const unsigned char* itmask;
  int ns;
  const int* st_itvar;
  double* swf;
  float* swf32;
  ZeroList zero;
  SiteVec v;     // direction (p null: none)
  double* v64;
  float* v32;    // may be null
};
void launch_swf(const DevLattice& L, const SwfArgs& a, hipStream_t st);
int launch_free_energy(const DevLattice& L, const SysParams& sp, const double* phi, const double* phi_m,
                       const double* rho, const double* swf, const double* u, const double* molscal,
                       double* partial, hipStream_t st);
int launch_grand_potential(const DevLattice& L, const SysParams& sp, const double* phi, const double* phi_m,
                           const double* rho, const double* swf, const double* molscal, const double* phib_state,
                           const double* cbulk, double* partial, hipStream_t st);
void launch_sum_partials(const double* partial, int n, double* out, hipStream_t st);

// range_restricted molecules (SF_Copol1stO.cpp:1246-1280): phi_m of the used
// states summed over the interior sites of the box lo..hi (partial sums per
// block), then C = phi_range / sum into the molecule's scalars (pref, ln C,
// phi_b = N C) and phi_m *= C
struct RangeBox {
  int lo[3], hi[3];
};
int launch_range_sum(const DevLattice& L, RangeBox box, unsigned uses, int ns, const double* phi_m, double* partial,
                     hipStream_t st);
void launch_range_scale(const DevLattice& L, unsigned uses, int ns, const double* partial, int nparts,
                        double phi_range, int N, double* scal, double* phi_m, hipStream_t st);

}  // namespace sfx

// sfx_block3.h -- several propagator ranks per launch on 3-D simple-cubic and FCC
// lattices and on 2-D ones (temporal blocking through LDS tiles).
#pragma once

#include <utility>
#include <vector>

#include "sfx_kernels.h"

namespace sfx {

// ranks per launch at most. Four rather than two: a launch of the 64^3 melt
// costs 4-6 us before and after its ranks (dispatch, the region's loads, the
// maximum), which two ranks pay twice. FP32 tangents, two chains: 14.4 / 16.2 us
// (forward / composing) for four ranks, 8.7 / 11.0 us for two; FP64 at 128^3:
// 65 / 113 us against 32 / 64 us, the region read half as often.
constexpr int kB3Ranks = 4;
constexpr int kB2Ranks = 8;        // on a 2-D lattice (sfx_block2.hip)
constexpr int kBRanks = kB2Ranks;  // the most of any
// ranks per launch at most of a variant (FP64 tangents in 3-D: four would need
// 87 KB of LDS, one workgroup per CU; by twos a product at 52 x 52 x 53, N = 60,
// takes 469 us, rank by rank and with the base swept first 974)
inline int block_ranks(const DevLattice& L, bool tangent, bool fp64) {
  return L.grad == 2 ? kB2Ranks : tangent && fp64 ? 2 : kB3Ranks;
}

// Ranks s0+1 .. s0+nr of one chain, all of one segment state.
template <typename T>
struct B3Args {
  const T* in;                 // rank s0 (stored scale)
  const T* din;                // its tangent (tangent sweeps)
  const T* g;                  // SWF of the state
  const T* v;                  // tangent direction of the state
  T* out[kBRanks];            // where rank s0+k goes (nullptr: not kept)
  T* dout[kBRanks];
  const T* pair[kBRanks];     // composition partner of rank s0+k
  const T* dpair[kBRanks];
  T* acc;                      // accumulator of the state (phi, or dphi for tangents)
  T* bacc;                     // tangent sweeps: phi's accumulator too, unless the base has been swept (nullptr)
  int nr;
  // FP32 log-scaling: the input is divided by max(rank s0) (maxv[s0]) and
  // every rank by the lattice maximum of g (gmax), in two dimensions by the
  // power of two above each; lnv[s] is the log of the
  // divisor accumulated up to rank s, lnpair[pidx[k]] that of the partner
  unsigned* maxv;
  double* lnv;
  const double* lnpair;
  const double* ref;
  const unsigned* gmax;        // step-max slots of the state's lattice maximum of g
  unsigned* low;               // set when rank s0 has decayed too far (low_input)
  bool carried;                // rank s0 carries kBlockScale: it comes out of a blocked launch
  int s0;
  int pidx[kBRanks];
};

// One launch advancing up to two independent chains (the forward and the
// backward chain of a molecule): workgroups [0, nb) take chain 0, [nb, 2 nb)
// chain 1. Both run the same kernel variant (tangent / scaled / connect).
template <typename T>
struct B3Launch {
  B3Args<T> a[2];
  int nchains;
};

// Splits chain steps a..b (ascending) into launches: a launch ends at a grid
// line ((step - g0 + 1) % grid == 0), before a step of another segment state, or
// before a step that split() marks. f(first, last) per launch. The
// grid makes the partition of any stretch that starts on a grid line equal
// to that of the whole chain, so a recomputed stretch reproduces it bit for bit.
template <class State, class Split, class F>
void chain_blocks(int a, int b, int g0, State state, Split split, F f, int grid) {
  int s = a;
  while (s <= b) {
    int e = s;
    while (e < b && (e + 1 - g0) % grid != 0 && state(e + 1) == state(s) && !split(e + 1)) e++;
    f(s, e);
    s = e + 1;
  }
}

// the launches of chain_blocks(a, b, g0, state, no extra splits) as a list
template <class State>
std::vector<std::pair<int, int>> chain_launches(int a, int b, int g0, State state, int grid) {
  std::vector<std::pair<int, int>> out;
  chain_blocks(
      a, b, g0, state, [](int) { return false; }, [&](int s, int e) { out.emplace_back(s, e); }, grid);
  return out;
}

// true when the blocked sweep applies: 3-D simple cubic or FCC, first order, every
// side at least kB3Ranks + 1 layers (one reflection reaches the interior)
bool block3_ok(const DevLattice& L);
// true when the blocked sweep of 2-D lattices applies: first order, its own adjoint
bool block2_ok(const DevLattice& L);

// ev0/ev1 (optional): timing events the dispatch records at kernel start and end
template <typename T>
void launch_block3(const DevLattice& L, const B3Launch<T>& la, bool tangent, bool scaled, bool connect,
                   hipStream_t st, hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr);

template <typename T>
void launch_block2(const DevLattice& L, const B3Launch<T>& la, bool tangent, bool scaled, bool connect,
                   hipStream_t st, hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr);

// max over the interior of each state's FP32 SWF, into step-max slots
// gmax + t * kStepWords (zeroed here)
// zeroed: gmax[0, ns * kStepWords) is already 0 on st (launch_swf can clear it)
void launch_gmax(const DevLattice& L, const float* swf32, int ns, unsigned* gmax, hipStream_t st,
                 bool zeroed = false);

}  // namespace sfx

// sfx_block2.hip -- temporally blocked propagator ranks on 2-D lattices, flat
// and cylindrical: one launch advances a chain (or the two chains of a
// middle-out sweep) by up to eight ranks.
//
// A 2-D lattice of some ten thousand sites is a few microseconds of work per
// rank for a fraction of the chip, so a launch per rank is all dispatch: 78
// launches of 3.6 us (FP64), 156 of 5.3 us for an FP32 product, at 64 x 128
// and N = 40. Here a workgroup of six waves owns 8 x 48 sites and holds them
// widened by eight on every side, 24 x 64: a wave has four x rows, a lane one
// y. The y neighbours come from the next lanes by a wave shift, the x
// neighbours from the wave's own registers and, at its first and last row,
// from the neighbouring waves through LDS: one barrier per rank. Sites behind
// a bound are images of interior sites (their g and radial weights mirrored
// with them), behind a surface 0.
//   G_k(r) = g(r) A[G_{k-1}](r)  (Lat2DFlat1stO.cpp:31-52, Lat2DCyl1stO.cpp:16-39)
// Composition and tangents are those of sfx_block3.hip, and so is FP32 scaling
// but that its divisors are powers of two: of eight ranks, up to eight decay
// between renormalisations (kLowMax).
//
// What bounds it: the ranks' dependent operations and barriers, and the
// launch's loads and dispatch before them. At 64 x 128 a launch of eight ranks
// takes 6.3 / 9.9 us (forward / composing, both chains) in FP64 and 9.2 / 12.3
// us for an FP32 product; with it the N = 40 residual went from 376 to 154 us and
// the product from 978 to 217 us (100 and 143 us since the launches around it were
// fused). Why eight ranks: the widened tile costs four times the tile's work,
// which the idle chip has to spare, and a launch's fixed 4 us are paid an eighth
// as often.
#include <hip/hip_ext.h>

#include "sfx_block3.h"
#include "sfx_device.h"

namespace sfx {

constexpr int kB2H = kB2Ranks;                        // widening
constexpr int kB2Rows = 4, kB2Waves = 6;              // x rows per wave, waves
constexpr int kB2X = kB2Rows * kB2Waves - 2 * kB2H;   // owned rows: 8
constexpr int kB2Y = 64 - 2 * kB2H;                   // owned columns: 48
constexpr int kB2Threads = 64 * kB2Waves;
static_assert(kB2H % kB2Rows == 0 && kB2X % kB2Rows == 0, "a wave's rows are all owned or none");

bool block2_ok(const DevLattice& L) {
  // a curved lattice with a mirror2 side or radial wrap-around (layers of
  // different volumes exchange through one weight each): its sweep is not its own
  // adjoint, so the two chains of a middle-out sweep would not agree
  bool adjoint = !L.periodic[0];
  for (int k = 0; k < 2; k++) adjoint &= !L.mirror2_1[k] && !L.mirror2_2[k];
  return L.grad == 2 && L.order == 1 && (!L.curved || adjoint);
}

// The factor 2^-e that a step maximum m stands for, 2^(e-1) <= m < 2^e, and
// ln = e ln 2 (m = 0 or NaN: 1 and 0). A power of two divides without rounding;
// 1 / m rounds every word, the SWF's in each rank of a launch the same way,
// which over eight ranks a launch doubled the error of an FP32 product
// (64 x 128 pore, N = 40: 1.7e-7 against 9e-8).
__device__ __forceinline__ float pow2_scale(float m, double& ln) {
  if (!(m > 0.f)) {
    ln = 0.0;
    return 1.f;
  }
  const int e = min((int)(__float_as_uint(m) >> 23) - 126, 126);
  ln = (double)e * 0.69314718055994530942;
  return __uint_as_float((unsigned)(127 - e) << 23);
}

// interior coordinate of which c is the image (every side has at least two
// layers, so the reflections end); 0 behind a surface. flip: an odd
// number of reflections
__device__ __forceinline__ int image(int c, int n, int lo, int hi, bool& flip) {  // 0 surface 1 mirror1 2 mirror2 3 periodic
  flip = false;
  while (c < 1 || c > n) {
    const int how = c < 1 ? lo : hi;
    if (how == 0) return 0;
    if (how == 3) {
      c += c < 1 ? n : -n;
    } else {
      flip = !flip;
      c = c < 1 ? how - c : 2 * n + 2 - how - c;
    }
  }
  return c;
}

// a word from the lane below / above (0 beyond the wave)
template <typename T, int CTRL>
__device__ __forceinline__ T shifted(T v) {
  if constexpr (sizeof(T) == 4) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
  } else {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
  }
}

template <typename T, bool TANGENT, bool SCALED, bool CONNECT>
__global__ void __launch_bounds__(kB2Threads) k_block2(DevLattice L, B3Launch<T> la, int nb) {
  constexpr int R = kB2Rows;
  const int chain = (int)blockIdx.x >= nb ? 1 : 0;
  const int bl = (int)blockIdx.x - chain * nb;
  const B3Args<T>& a = la.a[chain];
  // first and last row of every wave, two buffers; the tangent's behind them
  __shared__ T rows[2][TANGENT ? 2 : 1][kB2Waves][2][64];
  __shared__ float red[kB2Waves], scl[2];
  __shared__ T cfac[kB2Ranks];

  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nr = a.nr;

  // the maxima and logs of earlier launches first (sfx_block3.hip)
  float ma = 0.f, mb = 0.f;
  double lnv0 = 0.0, lnp = 0.0, lref = 0.0;
  int power = 0;  // of this lane's composition factor
  if constexpr (SCALED) {
    if (wave == 0) {
      ma = __uint_as_float(a.maxv[(long long)a.s0 * kStepWords + lane * kSlotStride]);
      mb = __uint_as_float(a.gmax[lane * kSlotStride]);
      lnv0 = a.lnv[a.s0];
      if constexpr (CONNECT) {
        int pi = a.pidx[0];
#pragma unroll
        for (int k = 1; k < kB2Ranks; k++)
          if (lane == k) pi = a.pidx[k];
        if (lane < nr) lnp = a.lnpair[pi];
        lref = *a.ref;
        power = (int)a.ref[MS_POW - MS_REF] - kBlockPower * (pi >= 2 ? 2 : 1);
      }
    }
  }

  const int nby = (L.ny + kB2Y - 1) / kB2Y;
  const int by = bl % nby, bx = bl / nby;
  const int x0 = 1 + bx * kB2X, y0 = 1 + by * kB2Y;
  auto bound = [](int surf, int m2, int per) { return surf ? 0 : per ? 3 : m2 ? 2 : 1; };
  const int ylo = bound(L.surf1[1], L.mirror2_1[1], L.periodic[1]), yhi = bound(L.surf2[1], L.mirror2_2[1], L.periodic[1]);
  const int xlo = bound(L.surf1[0], L.mirror2_1[0], L.periodic[0]), xhi = bound(L.surf2[0], L.mirror2_2[0], L.periodic[0]);
  bool flip;
  const int y = image(y0 - kB2H + lane, L.ny, ylo, yhi, flip);
  // this wave's rows are owned, and this lane's column
  const bool rows_owned = wave * R >= kB2H && wave * R < kB2H + kB2X;
  const bool owner = rows_owned && lane >= kB2H && lane < kB2H + kB2Y && y0 + lane - kB2H <= L.ny;

  T G[R], g[R], D[TANGENT ? R : 1], v[TANGENT ? R : 1], lm[R], lp[R];
  unsigned px[R];
  bool in[R];  // an owned row inside the lattice
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int xr = x0 - kB2H + wave * R + r;
    const int x = image(xr, L.nx, xlo, xhi, flip);
    in[r] = xr <= L.nx;
    px[r] = (unsigned)x * (unsigned)L.jx;
    const bool some = x > 0 && y > 0;
    G[r] = some ? (a.in + px[r])[y] : T(0);
    g[r] = some ? (a.g + px[r])[y] : T(0);
    if constexpr (TANGENT) {
      D[r] = some ? (a.din + px[r])[y] : T(0);
      v[r] = some ? (a.v + px[r])[y] : T(0);
    }
    lm[r] = lp[r] = T(0);
    if (L.curved) {
      lm[r] = T(flip ? L.lp[x] : L.lm[x]);
      lp[r] = T(flip ? L.lm[x] : L.lp[x]);
    }
  }

  double ln_base = 0.0, lng = 0.0;
  if constexpr (SCALED) {
    if (wave == 0) {
      for (int o = 32; o > 0; o >>= 1) {
        ma = fmaxf(ma, __shfl_xor(ma, o, 64));
        mb = fmaxf(mb, __shfl_xor(mb, o, 64));
      }
      if (a.carried) ma *= kBlockDown;
      if (lane == 0 && bl == 0 && low_input(ma, a.carried)) *a.low = 1u;
      double lna;
      const float sa = pow2_scale(ma, lna), sb = pow2_scale(mb, lng);
      if (lane == 0) {
        scl[0] = sa * (a.carried ? 1.f : kBlockScale);
        scl[1] = sb;
      }
      if (CONNECT || bl == 0) {
        ln_base = lnv0 + lna;
        if constexpr (CONNECT) {
          const double cf = lane < nr ? ldexp(exp(ln_base + (lane + 1) * lng + lnp - lref), power) : 1.0;
          if (lane < kB2Ranks) cfac[lane] = (T)cf;
        }
      }
    }
    __syncthreads();
    const T in_scale = (T)scl[0], ginv = (T)scl[1];
#pragma unroll
    for (int r = 0; r < R; r++) {
      G[r] *= in_scale;
      g[r] *= ginv;
      if constexpr (TANGENT) D[r] *= in_scale;
    }
  }

  T acc[CONNECT ? R : 1], bacc[CONNECT && TANGENT ? R : 1];
  if constexpr (CONNECT) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      acc[r] = T(0);
      if constexpr (TANGENT) bacc[r] = T(0);
    }
  }
  const T l1 = T(L.l1), l0 = T(L.l0_2d), l1x = T(L.l1x), l1y = T(L.l1y);
  // A[P] of the wave's rows, up and dn the rows before and behind them
  auto average = [&](const T (&P)[R], T up, T dn, T (&A)[R]) __attribute__((always_inline)) {
    T xm = up;
#pragma unroll
    for (int r = 0; r < R; r++) {
      const T b = P[r], xp = r + 1 < R ? P[r + 1 < R ? r + 1 : r] : dn;
      const T ya = shifted<T, 0x138>(b), yc = shifted<T, 0x130>(b);
      A[r] = L.curved ? step2_curved(lm[r], lp[r], l1, xm, xp, ya, yc, b) : step2_flat(l0, l1x, l1y, xm, xp, ya, yc, b);
      xm = b;
    }
  };
#pragma unroll 1
  for (int k = 1; k <= nr; k++) {
    T pr[CONNECT ? R : 1], dpr[CONNECT && TANGENT ? R : 1];
    if constexpr (CONNECT) {
      if (owner) {  // in flight through the exchange
#pragma unroll
        for (int r = 0; r < R; r++) {
          pr[r] = (a.pair[k - 1] + px[r])[y];
          if constexpr (TANGENT) dpr[r] = (a.dpair[k - 1] + px[r])[y];
        }
      }
    }
    T(*const buf)[kB2Waves][2][64] = rows[k & 1];
    buf[0][wave][0][lane] = G[0];
    buf[0][wave][1][lane] = G[R - 1];
    if constexpr (TANGENT) {
      buf[TANGENT ? 1 : 0][wave][0][lane] = D[0];
      buf[TANGENT ? 1 : 0][wave][1][lane] = D[R - 1];
    }
    __syncthreads();
    const int wu = wave > 0 ? wave - 1 : 0, wd = wave + 1 < kB2Waves ? wave + 1 : wave;  // the outer rows: never reach the tile
    T A[R];
    average(G, buf[0][wu][1][lane], buf[0][wd][0][lane], A);
    if constexpr (TANGENT) {
      T dA[R];
      average(D, buf[TANGENT ? 1 : 0][wu][1][lane], buf[TANGENT ? 1 : 0][wd][0][lane], dA);
#pragma unroll
      for (int r = 0; r < R; r++) D[r] = g[r] * (dA[r] - v[r] * A[r]);
    }
#pragma unroll
    for (int r = 0; r < R; r++) G[r] = g[r] * A[r];
    if (owner) {
      T* const outk = a.out[k - 1];
      T* const doutk = TANGENT ? a.dout[k - 1] : nullptr;
      if (outk) {
#pragma unroll
        for (int r = 0; r < R; r++)
          if (in[r]) {
            (outk + px[r])[y] = G[r];
            if constexpr (TANGENT) (doutk + px[r])[y] = D[r];
          }
      }
      if constexpr (CONNECT) {
        const T cf = SCALED ? cfac[k - 1] : T(1);
#pragma unroll
        for (int r = 0; r < R; r++) {
          if constexpr (TANGENT) {
            acc[r] += (D[r] * pr[r] + G[r] * dpr[r]) * cf;
            bacc[r] += G[r] * pr[r] * cf;
          } else {
            acc[r] += G[r] * pr[r] * cf;
          }
        }
      }
    }
  }

  if constexpr (CONNECT) {
    if (owner) {
#pragma unroll
      for (int r = 0; r < R; r++)
        if (in[r]) {
          (a.acc + px[r])[y] += acc[r];
          if constexpr (TANGENT)
            if (a.bacc) (a.bacc + px[r])[y] += bacc[r];
        }
    }
  }
  if constexpr (SCALED) {
    float m = 0.f;
    if (owner) {
#pragma unroll
      for (int r = 0; r < R; r++)
        if (in[r]) m = fmaxf(m, (float)G[r]);
    }
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    if (lane == 0) red[wave] = m;
    __syncthreads();
    if (t == 0) {
      for (int i = 1; i < kB2Waves; i++) m = fmaxf(m, red[i]);
      put_step_max(a.maxv, a.s0 + nr, m);
      if (bl == 0)
        for (int k = 1; k <= nr; k++) a.lnv[a.s0 + k] = ln_base + k * lng;
    }
  }
}

template <typename T, bool TG, bool SC, bool CN>
static void b2_launch(const DevLattice& L, const B3Launch<T>& a, unsigned nb, hipStream_t st, hipEvent_t ev0,
                      hipEvent_t ev1) {
  hipExtLaunchKernelGGL((k_block2<T, TG, SC, CN>), dim3(nb * (unsigned)a.nchains), dim3(kB2Threads), 0, st, ev0, ev1,
                        0u, L, a, (int)nb);
}

template <typename T>
void launch_block2(const DevLattice& L, const B3Launch<T>& a, bool tangent, bool scaled, bool connect,
                   hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
  for (int c = 0; c < a.nchains; c++)
    SFX_REQUIRE(a.a[c].nr >= 1 && a.a[c].nr <= kB2Ranks, SFX_E_INVALID, "blocked launch of 1..8 ranks");
  const unsigned nb = (unsigned)(((L.nx + kB2X - 1) / kB2X) * ((L.ny + kB2Y - 1) / kB2Y));
#define B2(TG, SC, CN) b2_launch<T, TG, SC, CN>(L, a, nb, st, ev0, ev1)
  if constexpr (sizeof(T) == 4) {  // FP32 sweeps are scaled, FP64 ones are not
    SFX_REQUIRE(scaled, SFX_E_INVALID, "FP32 blocked sweeps are scaled");
    if (tangent) { if (connect) B2(true, true, true); else B2(true, true, false); }
    else { if (connect) B2(false, true, true); else B2(false, true, false); }
  } else {
    SFX_REQUIRE(!scaled, SFX_E_INVALID, "FP64 blocked sweeps are not scaled");
    if (tangent) { if (connect) B2(true, false, true); else B2(true, false, false); }
    else { if (connect) B2(false, false, true); else B2(false, false, false); }
  }
#undef B2
  SFX_HIP(hipGetLastError());
}
template void launch_block2<float>(const DevLattice&, const B3Launch<float>&, bool, bool, bool, hipStream_t,
                                   hipEvent_t, hipEvent_t);
template void launch_block2<double>(const DevLattice&, const B3Launch<double>&, bool, bool, bool, hipStream_t,
                                    hipEvent_t, hipEvent_t);

}  // namespace sfx

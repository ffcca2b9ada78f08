// sfx_block3.hip -- temporally blocked propagator ranks on 3-D simple-cubic and
// FCC lattices: one launch advances a chain by up to four ranks.
//
// A workgroup owns an 8 x 8 x 16 output tile. It loads the previous rank and
// the state's SWF on the tile widened by the number of ranks nr in every
// direction (a lattice with bounds extends by periodic wrap or by reflection,
// mirror1 about the face and mirror2 about the first layer, which is what the
// per-rank halo copies of Lat3D.cpp:892-1562 amount to), then computes rank k
// on the tile widened by nr - k:
//   G_k(r) = g(r) (1/6) sum_6 G_{k-1}(r + e)            (Lat3D1stO.cpp:53-260)
//   dG_k(r) = g(r) ((1/6) sum_6 dG_{k-1} - v(r) (1/6) sum_6 G_{k-1})
// (FCC: (1/12) sum_12 over the edge neighbours, Lat3DFCC1stO.cpp:77-89; at 50 x
// 41 x 63 four FP64 ranks take 10.3 / 11.2 us where one took 3.7 / 4.0)
// Two threads hold one (y, z) column of the widened tile, half of its x planes
// each, in registers, with g (and v) beside them: the x neighbours are
// registers, the y and z neighbours come from LDS, where every rank is
// exchanged, at addresses that differ from the thread's own by constants. The
// owned sites of every rank are stored and composed from those registers,
// acc += G_k G_pair c_k (ConnectG, Lat3D1stO.cpp:299-312; tangent
// dacc += (dG_k G_pair + G_k dG_pair) c_k), and acc goes to HBM once.
//
// What bounds it: at 64^3 a launch is one chain of waits, 5-10k of 22k cycles on
// the region's loads (rows of 96 bytes touch 1.7 lines, near the L2's rate), 3k
// on the scale factors and the first barrier, 11k in four ranks; 12% fewer loads
// and instructions changed nothing. At 128^3 it is the region's reads and HBM.
// The form before gave each thread of a 1024-thread workgroup one site at a time
// and spent most of its instructions on the divisions that found it. Four ranks
// of two chains at 64^3, FP32: 17.5 / 21.5 us then, 9.0 / 11.1 us now (forward /
// composing), tangents 25 / 29 us then, 14.4 / 18.0 us now, base and tangent
// composed together; FP64 at 128^3: 122 / 160 us then, 63 / 112 us now. One
// thread per column (twice the planes each) took 11.7 / 14.7 us in FP32.
//
// FP32 scaling: the input is divided by max(rank s0) and every rank by the
// lattice maximum of g, so no rank exceeds 1 and at most nr ranks decay
// between renormalisations; the logs of the divisors go to lnv. Stored ranks and
// maxima carry a factor 2^32, and a launch whose ranks decay too far says so
// (kLowMax).
#include <hip/hip_ext.h>

#include <algorithm>

#include "sfx_block3.h"
#include "sfx_device.h"

namespace sfx {

constexpr int kTX = 8, kTY = 8, kTZ = 16;  // (x: or 2 kTX, see b3_launch_h)
static_assert(kTY % 2 == 0, "rows are numbered in pairs outside the tile");
constexpr int kH = kB3Ranks;  // largest widening: the lattice-side bound of block3_ok
// the tile widened by H layers; one (y, z) column of it is two threads, each
// with px of its x planes in registers
template <int H, int KIND, int TX = kTX>
struct B3Region {
  static constexpr int rx = TX + 2 * H, ry = kTY + 2 * H, rz = kTZ + 2 * H;
  static constexpr int px = rx / 2;
  static constexpr int half = (ry * rz + 63) / 64 * 64;  // threads of one half
  static constexpr int threads = 2 * half;
  // LDS words of one rank: the planes from p0 to px - 1 of each half (on the
  // simple cubic lattice the outermost one is nobody's y or z neighbour), a row
  // and a word of padding below and above
  static constexpr int p0 = KIND == ST_3D_SC ? 1 : 0, planes = px - p0, pad = rz + 1;
  static constexpr int words = 2 * planes * half + 2 * pad;
};
// two LDS buffers (one barrier per rank) where they leave room for three
// workgroups per CU, else one buffer and two barriers
template <typename T, bool TANGENT, int H, int KIND, int TX = kTX>
constexpr bool b3_double() {
  return 2 * (TANGENT ? 2 : 1) * B3Region<H, KIND, TX>::words * (int)sizeof(T) <= 53 * 1024;
}
template <typename T, bool TANGENT, int H, int KIND, int TX = kTX>
constexpr int b3_lds() {
  return (b3_double<T, TANGENT, H, KIND, TX>() ? 2 : 1) * (TANGENT ? 2 : 1) * B3Region<H, KIND, TX>::words * (int)sizeof(T);
}

bool block3_ok(const DevLattice& L) {
  return L.grad == 3 && (L.kind == ST_3D_SC || L.kind == ST_3D_FCC) && L.order == 1 && L.nx > kH && L.ny > kH && L.nz > kH;
}

// lattice coordinate c -> interior coordinate. Within kH of the lattice one
// wrap or reflection is exact (every side has more than kH layers); farther
// out (a tile hanging over the lattice's far edge) the value never reaches a
// tile site inside the lattice, and the coordinate is only clamped into range.
__device__ __forceinline__ int extend(int c, int n, int periodic, int m2lo, int m2hi) {
  if (c < 1) c = periodic ? c + n : (m2lo ? 2 - c : 1 - c);
  else if (c > n) c = periodic ? c - n : (m2hi ? 2 * n - c : 2 * n + 1 - c);
  return c < 1 ? 1 : (c > n ? n : c);
}

// float maximum over the workgroup; valid in thread 0
template <int NT>
__device__ __forceinline__ float block_max_f(float v, float* red) {
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float r = red[0];
  for (int i = 1; i < NT / 64; i++) r = fmaxf(r, red[i]);
  return r;
}

template <typename T, bool TANGENT, bool SCALED, bool CONNECT, int H, int KIND, int TX = kTX>
__global__ void __launch_bounds__((B3Region<H, KIND, TX>::threads)) k_block3(DevLattice L, B3Launch<T> la, int nb) {
  using R = B3Region<H, KIND, TX>;
  constexpr int PX = R::px, RX = R::rx, RZ = R::rz, NT = R::half;
  constexpr int OX = PX - H;  // owned planes of a half: its planes H..PX-1
  constexpr bool DB = b3_double<T, TANGENT, H, KIND, TX>();
  // chain of this workgroup and its tile number within that chain's grid
  const int chain = (int)blockIdx.x >= nb ? 1 : 0;
  const int bl = (int)blockIdx.x - chain * nb;
  const B3Args<T>& a = la.a[chain];
  __shared__ __align__(16) T lds[b3_lds<T, TANGENT, H, KIND, TX>() / sizeof(T)];
  __shared__ float red[R::threads / 64], scl[2];
  __shared__ T cfac[kB3Ranks];

  const int t = threadIdx.x, lane = t & 63;
  const int nr = a.nr;

  // the maxima and logs the scale factors build on were written by earlier
  // launches: the first wave asks for them before anything else, so that they
  // arrive before the region and are worked on while it is in flight
  float ma = 0.f, mb = 0.f;
  double lnv0 = 0.0, lnp = 0.0, lref = 0.0;
  int power = 0;  // of this lane's composition factor
  if constexpr (SCALED) {
    if (t < 64) {
      ma = __uint_as_float(a.maxv[(long long)a.s0 * kStepWords + lane * kSlotStride]);
      mb = __uint_as_float(a.gmax[lane * kSlotStride]);
      lnv0 = a.lnv[a.s0];
      if constexpr (CONNECT) {
        int pi = a.pidx[0];
#pragma unroll
        for (int k = 1; k < kB3Ranks; k++)
          if (lane == k) pi = a.pidx[k];
        if (lane < nr) lnp = a.lnpair[pi];
        lref = *a.ref;
        power = (int)a.ref[MS_POW - MS_REF] - kBlockPower * (pi >= 2 ? 2 : 1);
      }
    }
  }

  const int nbz = (L.nz + kTZ - 1) / kTZ, nby = (L.ny + kTY - 1) / kTY;
  // XCD-aware: each XCD takes a contiguous run of tiles (x-slabs), so the y / z
  // halos its tiles share stay in that XCD's L2
  int b = (int)xcd_tile(bl, nb);
  const int bz = b % nbz;
  b /= nbz;
  const int by = b % nby;
  const int bx = b / nby;
  const int x0 = 1 + bx * TX, y0 = 1 + by * kTY, z0 = 1 + bz * kTZ;  // tile origin (interior coords)

  // this thread's (y, z) column and its half of it: plane j of the lower half
  // is region plane j, of the upper half region plane RX-1-j, so that in both
  // plane j-1 lies outwards, j+1 inwards, rank k needs the planes j >= k, and
  // the planes H.. are owned where (y, z) lies in the tile and in the lattice
  const int half = __builtin_amdgcn_readfirstlane(t >= NT ? 1 : 0);
  const int c = t - half * NT;
  // rows of the region from the tile's outwards, so that whole waves have no
  // row left that a later rank needs: `row` is the wave's innermost
  const int ring = c / RZ, Z = c - ring * RZ;
  const int off = (ring - kTY) / 2;  // (threads past the last row keep a word of their own behind it)
  const int Y = ring < kTY ? H + ring : ring >= R::ry ? ring : ring & 1 ? H + kTY + off : H - 1 - off;
  const int row = __builtin_amdgcn_readfirstlane(ring);
  const bool owner = Y >= H && Y < H + kTY && Z >= H && Z < H + kTZ && y0 + Y - H <= L.ny && z0 + Z - H <= L.nz;
  const int yy = extend(y0 + Y - H, L.ny, L.periodic[1], L.mirror2_1[1], L.mirror2_2[1]);
  const int zz = extend(z0 + Z - H, L.nz, L.periodic[2], L.mirror2_1[2], L.mirror2_2[2]);
  const unsigned yz = (unsigned)(yy * L.MZ + zz);
  // plane offsets: one lane each, then into scalar registers
  const int xl = x0 - H + (half ? RX - 1 - lane : lane);
  const unsigned xoff =
      (unsigned)extend(xl, L.nx, L.periodic[0], L.mirror2_1[0], L.mirror2_2[0]) * (unsigned)L.jx;
  unsigned px[PX];
#pragma unroll
  for (int j = 0; j < PX; j++) px[j] = (unsigned)__builtin_amdgcn_readlane((int)xoff, j);
  // owned plane j lies in the lattice
  auto inside = [&](int j) { return x0 + (half ? TX - 1 - (j - H) : j - H) <= L.nx; };

  // rank s0 (and its tangent), g (and v) of the column: the plane's offset is
  // uniform, the lane's is one 32-bit word
  T G[PX], g[PX], D[TANGENT ? PX : 1], v[TANGENT ? PX : 1];
#pragma unroll
  for (int j = 0; j < PX; j++) {
    G[j] = (a.in + px[j])[yz];
    if constexpr (TANGENT) D[j] = (a.din + px[j])[yz];
  }
#pragma unroll
  for (int j = 1; j < PX; j++) {
    g[j] = (a.g + px[j])[yz];
    if constexpr (TANGENT) v[j] = (a.v + px[j])[yz];
  }

  // scale factors of this launch: the FP64 logs and exponentials are evaluated
  // by the first wave alone (lanes 0 and 1 the logs of the two divisors, lane k
  // the composition factor of rank k + 1) while the region is in flight
  double ln_base = 0.0, lng = 0.0;
  if constexpr (SCALED) {
    if (t < 64) {
      for (int o = 32; o > 0; o >>= 1) {
        ma = fmaxf(ma, __shfl_xor(ma, o, 64));
        mb = fmaxf(mb, __shfl_xor(mb, o, 64));
      }
      if (a.carried) ma *= kBlockDown;
      if (lane == 0 && bl == 0 && low_input(ma, a.carried)) *a.low = 1u;
      if (!(ma > 0.f)) ma = 1.f;
      if (!(mb > 0.f)) mb = 1.f;
      if (lane == 0) {
        scl[0] = 1.f / ma * (a.carried ? 1.f : kBlockScale);
        scl[1] = 1.f / mb;
      }
      if (CONNECT || bl == 0) {
        const double lv = log((double)(lane == 1 ? mb : ma));
        ln_base = lnv0 + __shfl(lv, 0, 64);
        lng = __shfl(lv, 1, 64);
        if constexpr (CONNECT) {
          const double cf = lane < nr ? ldexp(exp(ln_base + (lane + 1) * lng + lnp - lref), power) : 1.0;
          if (lane < kB3Ranks) cfac[lane] = (T)cf;
        }
      }
    }
    __syncthreads();
    const T in_scale = (T)scl[0], ginv = (T)scl[1];
#pragma unroll
    for (int j = 0; j < PX; j++) {
      G[j] *= in_scale;
      if (j) g[j] *= ginv;
      if constexpr (TANGENT) D[j] *= in_scale;
    }
  }

  T acc[CONNECT ? OX : 1], bacc[CONNECT && TANGENT ? OX : 1];
  if constexpr (CONNECT) {
#pragma unroll
    for (int i = 0; i < OX; i++) {
      acc[i] = T(0);
      if constexpr (TANGENT) bacc[i] = T(0);
    }
  }
  // LDS word of this column's plane p0, and of the other half's
  const unsigned pos = (unsigned)(R::pad + Y * RZ + Z);
  const unsigned own = pos + (unsigned)(half * R::planes * NT), other = pos + (unsigned)((1 - half) * R::planes * NT);
  // the sum over the stencil at plane j, from the rank in E (registers) and buf:
  // simple cubic six faces; FCC the in-plane diagonals and the faces of the
  // planes before and behind, whose sums the caller rolls on
  auto faces = [&](const T* buf, unsigned o) __attribute__((always_inline)) {
    return buf[o - RZ] + buf[o + RZ] + buf[o - 1] + buf[o + 1];
  };
  auto diagonals = [&](const T* buf, unsigned o) __attribute__((always_inline)) {
    return buf[o - RZ - 1] + buf[o - RZ + 1] + buf[o + RZ - 1] + buf[o + RZ + 1];
  };
  // `out`: what plane j takes from the next plane outwards, rolled on
  auto stencil_sum = [&](const T (&E)[PX], const T* buf, int j, T& out, T& here) __attribute__((always_inline)) {
    const unsigned o = own + (j - R::p0) * NT;
    if constexpr (KIND == ST_3D_SC) {
      const T in = j + 1 < PX ? E[j + 1 < PX ? j + 1 : j] : buf[other + (R::planes - 1) * NT];
      const T s = (out + in + buf[o - RZ] + buf[o + RZ] + buf[o - 1] + buf[o + 1]) * T(1.0 / 6.0);
      out = E[j];
      return s;
    } else {
      const T in = faces(buf, j + 1 < PX ? o + NT : other + (R::planes - 1) * NT);
      const T s = (out + in + diagonals(buf, o)) * T(1.0 / 12.0);
      out = here;
      here = in;
      return s;
    }
  };
#pragma unroll
  for (int k = 1; k <= H; k++) {
    if (k <= nr) {
      // the partner values of this rank, in flight through the exchange
      T pr[CONNECT ? OX : 1], dpr[CONNECT && TANGENT ? OX : 1];
      if constexpr (CONNECT) {
        if (owner) {
#pragma unroll
          for (int i = 0; i < OX; i++) {
            pr[i] = (a.pair[k - 1] + px[H + i])[yz];
            if constexpr (TANGENT) dpr[i] = (a.dpair[k - 1] + px[H + i])[yz];
          }
        }
      }
      T* const buf = lds + (DB && (k & 1) ? (TANGENT ? 2 : 1) * R::words : 0);
      T* const dbuf = buf + R::words;
      if (!DB && k > 1) __syncthreads();  // the previous rank's reads are done
      const int rows = kTY + 2 * (nr - k);  // rows that rank k is needed on
      if (row < rows + 2) {
#pragma unroll
        for (int j = k - 1 + R::p0; j < PX; j++) {
          buf[own + (j - R::p0) * NT] = G[j];
          if constexpr (TANGENT) dbuf[own + (j - R::p0) * NT] = D[j];
        }
      }
      __syncthreads();
      if (row < rows) {
        // what plane k takes from plane k - 1, and on FCC what plane k + 1 takes from k
        T out = G[k - 1], dout = TANGENT ? D[k - 1] : T(0), here = T(0), dhere = T(0);
        if constexpr (KIND != ST_3D_SC) {
          out = faces(buf, own + (k - 1) * NT);
          here = faces(buf, own + k * NT);
          if constexpr (TANGENT) {
            dout = faces(dbuf, own + (k - 1) * NT);
            dhere = faces(dbuf, own + k * NT);
          }
        }
#pragma unroll
        for (int j = k; j < PX; j++) {
          const T s = stencil_sum(G, buf, j, out, here);
          G[j] = g[j] * s;
          if constexpr (TANGENT) {
            const T ds = stencil_sum(D, dbuf, j, dout, dhere);
            D[j] = g[j] * (ds - v[j] * s);
          }
        }
      }
      // the owned tile sites of rank k: store and compose
      if (owner) {
        T* const outk = a.out[k - 1];
        T* const doutk = TANGENT ? a.dout[k - 1] : nullptr;
        if (outk) {
#pragma unroll
          for (int j = H; j < PX; j++)
            if (inside(j)) {
              (outk + px[j])[yz] = G[j];
              if constexpr (TANGENT) (doutk + px[j])[yz] = D[j];
            }
        }
        if constexpr (CONNECT) {
          const T cf = SCALED ? cfac[k - 1] : T(1);
#pragma unroll
          for (int i = 0; i < OX; i++) {
            if constexpr (TANGENT) {
              acc[i] += (D[H + i] * pr[i] + G[H + i] * dpr[i]) * cf;
              bacc[i] += G[H + i] * pr[i] * cf;
            } else {
              acc[i] += G[H + i] * pr[i] * cf;
            }
          }
        }
      }
    }
  }

  if constexpr (CONNECT) {
    if (owner) {
#pragma unroll
      for (int i = 0; i < OX; i++)
        if (inside(H + i)) {
          (a.acc + px[H + i])[yz] += acc[i];
          if constexpr (TANGENT)
            if (a.bacc) (a.bacc + px[H + i])[yz] += bacc[i];
        }
    }
  }
  if constexpr (SCALED) {
    T mloc = T(0);
    if (owner) {
#pragma unroll
      for (int j = H; j < PX; j++)
        if (inside(j)) mloc = mloc > G[j] ? mloc : G[j];
    }
    const float m = block_max_f<R::threads>((float)mloc, red);
    if (t == 0) {
      put_step_max(a.maxv, a.s0 + nr, m);
      if (bl == 0)
        for (int k = 1; k <= nr; k++) a.lnv[a.s0 + k] = ln_base + k * lng;
    }
  }
}

static unsigned b3_tiles(const DevLattice& L, int tx) {
  return (unsigned)(((L.nx + tx - 1) / tx) * ((L.ny + kTY - 1) / kTY) * ((L.nz + kTZ - 1) / kTZ));
}
template <typename T, bool TG, bool SC, bool CN, int H, int KIND, int TX = kTX>
static void b3_launch(const DevLattice& L, const B3Launch<T>& a, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
  static_assert(b3_lds<T, TG, H, KIND, TX>() <= 64 * 1024, "static LDS");
  const unsigned nb = b3_tiles(L, TX);
  // with events: recorded by the dispatch itself at kernel start and end
  hipExtLaunchKernelGGL((k_block3<T, TG, SC, CN, H, KIND, TX>), dim3(nb * (unsigned)a.nchains),
                        dim3(B3Region<H, KIND, TX>::threads), 0, st, ev0, ev1, 0u, L, a, (int)nb);
}
template <typename T, bool TG, bool SC, bool CN, int KIND>
static void b3_launch_h(int nr, const DevLattice& L, const B3Launch<T>& a, hipStream_t st, hipEvent_t ev0,
                        hipEvent_t ev1) {
  // launches of one or two ranks (a chain's ends, a change of the segment
  // state) load and compute a smaller region: 7.2 / 9.1 us instead of 14 / 16
  // at 75 x 61 x 90 in FP32
  if (nr <= 2) {
    b3_launch<T, TG, SC, CN, 2, KIND>(L, a, st, ev0, ev1);
    return;
  }
  // FP32 base ranks: a tile of 16 planes reads 4.5 times itself instead of 6,
  // from 3.5 workgroups of the smaller tile per CU on. With fewer the chip runs
  // out of waves (residuals at 40 x 42 x 45: 166 us by 8 planes, 193 by 16; at
  // 64 x 66 x 69 240 and 235; at 100 x 102 x 105 518 and 480). FP64 and
  // tangents, with twice the registers and LDS, are slower by it throughout
  // (100 x 102 x 105: 618 and 656 us in FP64, products 829 and 920 in FP32).
  if constexpr (!TG && sizeof(T) == 4 && KIND == ST_3D_SC) {
    if (b3_tiles(L, kTX) * (unsigned)a.nchains >= 896) {
      b3_launch<T, TG, SC, CN, kB3Ranks, KIND, 2 * kTX>(L, a, st, ev0, ev1);
      return;
    }
  }
  if constexpr (!(TG && sizeof(T) == 8)) b3_launch<T, TG, SC, CN, kB3Ranks, KIND>(L, a, st, ev0, ev1);
}

template <typename T>
void launch_block3(const DevLattice& L, const B3Launch<T>& a, bool tangent, bool scaled, bool connect,
                   hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
  SFX_REQUIRE(a.nchains == 1 || a.nchains == 2, SFX_E_INVALID, "a blocked launch advances one or two chains");
  if (L.grad == 2) {
    launch_block2<T>(L, a, tangent, scaled, connect, st, ev0, ev1);
    return;
  }
  int nr = 0;
  for (int c = 0; c < a.nchains; c++) {
    SFX_REQUIRE(a.a[c].nr >= 1 && a.a[c].nr <= block_ranks(L, tangent, sizeof(T) == 8), SFX_E_INVALID,
                "blocked launch of 1..4 ranks");
    nr = std::max(nr, a.a[c].nr);
  }
#define B3(TG, SC, CN)                                                         \
  (L.kind == ST_3D_FCC ? b3_launch_h<T, TG, SC, CN, ST_3D_FCC>(nr, L, a, st, ev0, ev1) \
                       : b3_launch_h<T, TG, SC, CN, ST_3D_SC>(nr, L, a, st, ev0, ev1))
  if constexpr (sizeof(T) == 4) {  // FP32 sweeps are scaled, FP64 ones are not
    SFX_REQUIRE(scaled, SFX_E_INVALID, "FP32 blocked sweeps are scaled");
    if (tangent) { if (connect) B3(true, true, true); else B3(true, true, false); }
    else { if (connect) B3(false, true, true); else B3(false, true, false); }
  } else {
    SFX_REQUIRE(!scaled, SFX_E_INVALID, "FP64 blocked sweeps are not scaled");
    if (tangent) { if (connect) B3(true, false, true); else B3(true, false, false); }
    else { if (connect) B3(false, false, true); else B3(false, false, false); }
  }
#undef B3
  SFX_HIP(hipGetLastError());
}

// max of each state's FP32 SWF over the interior: 64 workgroups per state,
// one atomic each on the state's word (zeroed first)
__global__ void k_gmax_zero(unsigned* gmax, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) gmax[i] = 0u;
}
__global__ void __launch_bounds__(256) k_gmax(DevLattice L, const float* __restrict__ swf32, unsigned* __restrict__ gmax) {
  const float* g = swf32 + (long long)blockIdx.y * L.M;
  float m = 0.f;
  for (long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x; q < L.V; q += (long long)gridDim.x * blockDim.x) {
    int x, y, z;
    interior_coords(L, q, x, y, z);
    m = fmaxf(m, g[sidx(L, x, y, z)]);
  }
  __shared__ float red[4];
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    put_step_max(gmax + (long long)blockIdx.y * kStepWords, 0, m);  // slot blockIdx.x mod kMaxSlots
  }
}

void launch_gmax(const DevLattice& L, const float* swf32, int ns, unsigned* gmax, hipStream_t st, bool zeroed) {
  const int n = ns * kStepWords;
  if (!zeroed) k_gmax_zero<<<grid1(n, 256), 256, 0, st>>>(gmax, n);
  const unsigned nb = (unsigned)std::min<long long>(256, std::max<long long>(1, L.V / 1024));
  k_gmax<<<dim3(nb, ns), 256, 0, st>>>(L, swf32, gmax);
  SFX_HIP(hipGetLastError());
}

template void launch_block3<float>(const DevLattice&, const B3Launch<float>&, bool, bool, bool, hipStream_t,
                                   hipEvent_t, hipEvent_t);
template void launch_block3<double>(const DevLattice&, const B3Launch<double>&, bool, bool, bool, hipStream_t,
                                    hipEvent_t, hipEvent_t);

}  // namespace sfx

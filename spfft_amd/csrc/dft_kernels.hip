// Matrix kernels of the sparse 3D FFT for gfx950: DFTs of any length as
// products with the cosine and sine matrices, on the FP64 matrix cores.
//
// A line of n points is summed over the pairs (r, n - r): with a_r = v_r +
// v_(n-r) and b_r = v_r - v_(n-r), outputs q and n - q are C_q +- i S_q, C_q =
// sum a_r cos(2 pi r q / n), S_q = sum b_r sin(2 pi r q / n). Two sums of at
// most n / 2 + 1 real products each, and only over the r that the sparse set
// holds (backward) or for the q it wants (forward). Even lengths halve that
// once more: backward, the sums over even and odd r give the outputs q, n/2 -
// q, n/2 + q and n - q together; forward, the inputs r and n/2 - r enter
// together, with the sign of q's parity. A wave computes 16 lines x 16 outputs
// with v_mfma_f64_16x16x4: lane l carries the data of line l % 16 and the
// cosine and sine of output l % 16, both at the r of its group l / 16.
//
// Data of either precision is summed in FP64 and rounded once per stage (the
// roots of FP32 tables are hi + lo).
//
// Why this and not an FFT: at these sizes a launch is bound by the chain that
// one wave walks through (a wave issues an instruction every 5 cycles, a kernel
// boundary costs 2 to 6 us), not by bandwidth. An FFT's passes are a chain of
// LDS round trips with index arithmetic between them and code for each length;
// the pruned sums are a short loop of 16 matrix instructions per 16 inputs and
// outputs, and one kernel serves every length. The y and x transforms of a plane
// run in one launch with no buffer between them, since a workgroup that owns a
// set of rows (columns) computes just their part of the first transform.
//
// Measured on the MI355X, FP64 C2C, spheres of radius 0.3 N, us per launch
// (plane kernels) or per backward + forward pair, against the kernels they
// replace: plane stage at 100^3 backward 20.7 -> 13.7, forward 20.5 -> 11.1
// (split stage); six bands of 60^3 26 -> 14, 24 -> 13; pair at 97^3 804 -> 39,
// 67^3 529 -> 27, 20^3 35 -> 18 (generic kernels; 14.7 with the sums over z in the
// plane kernel). At 100^3 the plane kernels
// write 16 MB in 13.7 us: bound by the two chains load - sum - store; the sums
// alone take 2.6 us of the matrix cores. From about 128 points on the sums
// dominate (their work per line grows with its length squared) and the fixed-
// length kernels win: 128^3 21.7 against 16.3, 256^3 402 against 137.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <type_traits>
#include <unordered_map>

#include "device_args.hpp"
#include "dft_kernels.hpp"
#include "fft_common.hpp"
#include "hip_check.hpp"
#include "profiling.hpp"

namespace spfft {

extern __shared__ __attribute__((aligned(16))) unsigned char spfft_lds_dft[];

namespace {

using namespace dev;
using namespace dft;

constexpr int kWave = 64;
constexpr int kZWaves = 4;
constexpr int kMaxWaves = 8;
constexpr size_t kLdsDefault = 64 * 1024;
constexpr size_t kLdsMax = 160 * 1024;

typedef double D4 __attribute__((ext_vector_type(4)));

// cos and sin of 2 pi r q / n
struct alignas(16) Trig {
  double c, s;
};

// ---- output slots (dft_kernels.hpp)

__host__ __device__ constexpr int out_types(int n) { return n % 2 == 0 ? 4 : 2; }
// Output index of (slot q, type t); -1 for none or one that another type names.
__device__ __forceinline__ int out_index(int n, int q, int t) {
  if (q >= out_slots(n)) return -1;
  if (n % 2 != 0) return t == 0 ? q : (q == 0 ? -1 : n - q);
  const int h = n / 2;
  if (q == 0) {
    if (t < 2) return t * h;
    return !packed_slot(n) ? -1 : (t == 2 ? n / 4 : h + n / 4);
  }
  if (4 * q == n && (t == 1 || t == 2)) return -1;
  return t == 0 ? q : (t == 1 ? h - q : (t == 2 ? h + q : n - q));
}

// ---- trig tables
//
// Per length a backward and a forward table in the order in which the lanes of
// a tile read them, [parity][round][lane group][slot]: 16 consecutive slots are
// one 256-byte segment, and any slot can start a tile. Entries past the last r
// are zero (lengths: dft_kernels.hpp).

#ifndef SPFFT_DFT_FLOAT
__global__ void k_dft_trig(Trig* tab, int n) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= out_table(n) + in_table(n)) return;
  const bool out = e < out_table(n);
  Trig* to = tab + e;
  if (!out) e -= out_table(n);
  const int np = parities(n);
  const int row = out ? out_row(n) : in_row(n);
  const int rounds = out ? out_rounds(n, n / 2) : in_rounds(n);
  const int slot = e % row, kl = e / row % 4, d = e / row / 4 % rounds, par = e / row / 4 / rounds;
  const int r = out ? np * (4 * d + kl) + par : 4 * d + kl;
  const int q = out || np == 1 ? slot : 2 * slot + par;
  if (r > (out ? n / 2 : last_quad(n))) {
    *to = Trig{0.0, 0.0};
    return;
  }
  // angle reduced to (-pi, pi], so that its argument has one rounding
  const int t = static_cast<int>(static_cast<long long>(r) * q % n);
  const int tt = 2 * t > n ? t - n : t;
  double sn, cs;
  sincospi(2.0 * static_cast<double>(tt) / static_cast<double>(n), &sn, &cs);
  // slot 0 of a packed length also carries output n / 4, in its odd sine sum
  if (out && par == 1 && q == 0 && packed_slot(n)) sn = r % 4 == 1 ? 1.0 : -1.0;
  *to = Trig{cs, sn};
}
#endif

__device__ __forceinline__ D4 mfma(double a, double b, D4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// data x trig product: lines are the tile's rows (DATA_ROWS) or its columns
template <bool DATA_ROWS>
__device__ __forceinline__ D4 product(double data, double trig, D4 c) {
  return DATA_ROWS ? mfma(data, trig, c) : mfma(trig, data, c);
}
// Row of a tile that lane l's accumulator element v holds.
__device__ __forceinline__ int tile_row(int lane, int v) { return lane / kTile + 4 * v; }

struct Cd {
  double re, im;
};
template <typename T>
__device__ __forceinline__ Cd wide(Cx<T> x) {
  return Cd{static_cast<double>(x.re), static_cast<double>(x.im)};
}
template <typename T>
__device__ __forceinline__ Cx<T> narrow(double re, double im) {
  return Cx<T>{static_cast<T>(re), static_cast<T>(im)};
}

// Inputs r and n - r of one line.
template <typename T>
struct Pair {
  Cx<T> p, m;
};

// Backward sums (sign +) of the slots q0 .. q0 + 15 of 16 lines over the inputs
// |r| <= k. fetch(r), r < out_span, gives the lane's line's inputs r and n - r:
// zero past k, and a zero second one when r = 0 or 2 r = n. REAL: hermitian
// input, given by p alone, and a real result. Roots (AHEAD: and inputs, when
// they come from memory) are held in two halves of CH rounds, one in flight while
// the other is summed.
template <typename T, bool EVEN, bool DATA_ROWS, bool REAL, int CH, bool AHEAD>
struct OutSums {
  static constexpr int NP = EVEN ? 2 : 1;  // parities of r, each with sums of its own
  D4 cr[NP] = {}, ci[NP] = {}, sr[NP] = {}, si[NP] = {};
  double xr = 0.0, xi = 0.0;  // packed slot 0: cosine sum of output n / 4

  // Roots of CH rounds.
  struct Roots {
    Trig t[CH * NP];
    // those of the rounds from d on (past the last one: its own again, not summed)
    __device__ __forceinline__ void load(int n, int rounds, int q0, const Trig* tab, int d) {
      const int lane = threadIdx.x % kWave;
      const int row = out_row(n);
      const int odd = out_rounds(n, n / 2) * 4 * row;  // the odd r's table
      const int at = lane / kTile * row + q0 + lane % kTile;
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        const int dd = min(d + u, rounds - 1);
#pragma unroll
        for (int j = 0; j < NP; ++j) t[NP * u + j] = at32(tab + j * odd + dd * 4 * row, at);
      }
    }
    // the first ones: ahead of run(), so that they arrive while the workgroup is
    // still getting the inputs ready
    __device__ __forceinline__ void first(int n, int k, int q0, const Trig* tab) {
      load(n, out_rounds(n, k), q0, tab, 0);
    }
  };

  template <typename Fetch>
  __device__ __forceinline__ void run(int n, int k, int q0, const Trig* tab, const Roots& head,
                                      Fetch&& fetch) {
    const int kl = threadIdx.x % kWave / kTile;
    Pair<T> in[AHEAD ? 2 : 1][CH * NP];
    Roots tr[2];
    tr[0] = head;
    const int rounds = out_rounds(n, k);
    const bool packed = q0 == 0 && packed_slot(n);
    auto load = [&](int half, int d) {
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        const int dd = min(d + u, rounds - 1);
#pragma unroll
        for (int j = 0; j < NP; ++j) in[half][NP * u + j] = fetch(NP * (4 * dd + kl) + j);
      }
    };
    auto sum = [&](int d, const Pair<T>* x, const Trig* t) {
#pragma unroll
      for (int j = 0; j < NP; ++j) {
        const Cd p = wide(x[j].p);
        if constexpr (REAL) {
          // a conjugate pair sums to a real number; r = 0 and n / 2 stand alone
          // (and the sine of their imaginary parts is zero)
          const int r = NP * (4 * d + kl) + j;
          const double ar = r == 0 || 2 * r == n ? p.re : 2.0 * p.re;
          cr[j] = product<DATA_ROWS>(ar, t[j].c, cr[j]);
          sr[j] = product<DATA_ROWS>(-2.0 * p.im, t[j].s, sr[j]);
          if (EVEN && j == 0 && packed) xr += ar;
        } else {
          const Cd m = wide(x[j].m);
          const double ar = p.re + m.re, ai = p.im + m.im;
          cr[j] = product<DATA_ROWS>(ar, t[j].c, cr[j]);
          ci[j] = product<DATA_ROWS>(ai, t[j].c, ci[j]);
          sr[j] = product<DATA_ROWS>(p.re - m.re, t[j].s, sr[j]);
          si[j] = product<DATA_ROWS>(p.im - m.im, t[j].s, si[j]);
          if (EVEN && j == 0 && packed) {
            xr += ar;
            xi += ai;
          }
        }
      }
    };
    if (AHEAD) load(0, 0);
#pragma unroll 1
    for (int d0 = 0; d0 < rounds; d0 += 2 * CH) {
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int dh = d0 + half * CH;
        if (dh + CH < rounds) {
          tr[1 - half].load(n, rounds, q0, tab, dh + CH);
          if (AHEAD) load(1 - half, dh + CH);
        }
        if (!AHEAD && dh < rounds) load(0, dh);
#pragma unroll
        for (int u = 0; u < CH; ++u) {
          if (dh + u < rounds) sum(dh + u, in[AHEAD ? half : 0] + NP * u, tr[half].t + NP * u);
        }
      }
    }
    if (EVEN && q0 == 0 && packed_slot(n)) {
      // the lane groups' even r alternate in sign (r / 2 = 4 d + kl)
      xr = (kl & 1) ? -xr : xr;
      xr += __shfl_xor(xr, 16);
      xr += __shfl_xor(xr, 32);
      if (!REAL) {
        xi = (kl & 1) ? -xi : xi;
        xi += __shfl_xor(xi, 16);
        xi += __shfl_xor(xi, 32);
      }
    }
  }

  // Outputs of accumulator element v, by type (real results in .re).
  __device__ __forceinline__ void outputs(int n, int q0, int v, Cd* o) const {
    if constexpr (EVEN) {
      const double c0r = cr[0][v] + cr[1][v], c1r = cr[0][v] - cr[1][v];
      const double s0r = sr[0][v] + sr[1][v], s1r = sr[1][v] - sr[0][v];
      if constexpr (REAL) {
        o[0].re = c0r + s0r;
        o[1].re = c1r + s1r;
        o[2].re = c1r - s1r;
        o[3].re = c0r - s0r;
      } else {
        const double c0i = ci[0][v] + ci[1][v], c1i = ci[0][v] - ci[1][v];
        const double s0i = si[0][v] + si[1][v], s1i = si[1][v] - si[0][v];
        o[0] = Cd{c0r - s0i, c0i + s0r};
        o[1] = Cd{c1r - s1i, c1i + s1r};
        o[2] = Cd{c1r + s1i, c1i - s1r};
        o[3] = Cd{c0r + s0i, c0i - s0r};
      }
      if (q0 == 0 && packed_slot(n)) {
        // slot 0: 0, n / 2, n / 4, 3n / 4
        const int lane = threadIdx.x % kWave, row = tile_row(lane, v);
        const bool zero = (DATA_ROWS ? lane % kTile : row) == 0;
        const double xvr = DATA_ROWS ? __shfl(xr, row) : xr;
        if constexpr (REAL) {
          o[0].re = zero ? c0r : o[0].re;
          o[1].re = zero ? c1r : o[1].re;
          o[2].re = zero ? xvr + sr[1][v] : o[2].re;
          o[3].re = zero ? xvr - sr[1][v] : o[3].re;
        } else {
          const double xvi = DATA_ROWS ? __shfl(xi, row) : xi;
          o[0] = zero ? Cd{c0r, ci[0][v] + ci[1][v]} : o[0];
          o[1] = zero ? Cd{c1r, ci[0][v] - ci[1][v]} : o[1];
          o[2] = zero ? Cd{xvr - si[1][v], xvi + sr[1][v]} : o[2];
          o[3] = zero ? Cd{xvr + si[1][v], xvi - sr[1][v]} : o[3];
        }
      }
    } else if constexpr (REAL) {
      o[0].re = cr[0][v] + sr[0][v];
      o[1].re = cr[0][v] - sr[0][v];
    } else {
      o[0] = Cd{cr[0][v] - si[0][v], ci[0][v] + sr[0][v]};
      o[1] = Cd{cr[0][v] + si[0][v], ci[0][v] - sr[0][v]};
    }
  }
};

// Inputs r, n - r, n/2 - r and n/2 + r of one line (the last two for even
// lengths only).
template <typename T>
struct Quad {
  Cx<T> p, m, hp, hm;
};
// Input quad r of a line whose storage element i is at(i). Past the last r (n /
// 4, or (n - 1) / 2 of an odd length) it repeats that one's.
template <bool EVEN, typename T, typename At>
__device__ __forceinline__ Quad<T> quad_at(int n, int r, At&& at) {
  Quad<T> x;
  const int rc = min(r, EVEN ? n / 4 : (n - 1) / 2);
  x.p = at(rc);
  x.m = at(rc == 0 ? 0 : n - rc);
  if constexpr (EVEN) {
    x.hp = at(n / 2 - rc);
    x.hm = at(n / 2 + rc);
  }
  return x;
}

// Forward sums (sign -): outputs q and n - q of the 16 slots j from j0 on, q =
// 2 j + par (even lengths) or j (odd ones), over quads r (see quad_at). An input
// that a quad names twice (r = 0: m and hm; 4 r = n: hp and hm) counts once; the
// roots of a repeated quad are zero. Halves as in OutSums.
template <typename T, bool EVEN, bool DATA_ROWS, bool REAL, int CH, bool AHEAD>
struct InSums {
  D4 cr = {}, ci = {}, sr = {}, si = {};
  Quad<T> in[AHEAD ? 2 : 1][CH];
  Trig tr[2][CH];

  template <typename Fetch>
  __device__ __forceinline__ void run(int n, int j0, int par, const Trig* tab, Fetch&& fetch) {
    const int lane = threadIdx.x % kWave;
    const int kl = lane / kTile;
    const int rounds = in_rounds(n);
    const int row = in_row(n);
    const int at = kl * row + j0 + lane % kTile;
    tab += par * rounds * 4 * row;
    const double sg = par ? -1.0 : 1.0;
    auto load_trig = [&](int half, int d) {
#pragma unroll
      for (int u = 0; u < CH; ++u) tr[half][u] = at32(tab + min(d + u, rounds - 1) * 4 * row, at);
    };
    auto load = [&](int half, int d) {
#pragma unroll
      for (int u = 0; u < CH; ++u) in[half][u] = fetch(4 * min(d + u, rounds - 1) + kl);
    };
    auto sum = [&](int d, const Quad<T>& x, const Trig& t) {
      const Cd zero = Cd{0.0, 0.0};
      const Cd p = wide(x.p);
      Cd m = wide(x.m), hp = zero, hm = zero;
      if constexpr (EVEN) {
        hp = wide(x.hp);
        hm = wide(x.hm);
      }
      if (d == 0 && kl == 0) m = hm = zero;
      if (EVEN && d == rounds - 1 && 4 * (4 * d + kl) == n) hp = hm = zero;
      double ar = p.re + m.re, br = p.re - m.re;
      if constexpr (EVEN) {
        ar += sg * (hp.re + hm.re);
        br -= sg * (hp.re - hm.re);
      }
      cr = product<DATA_ROWS>(ar, t.c, cr);
      sr = product<DATA_ROWS>(br, t.s, sr);
      if constexpr (!REAL) {
        double ai = p.im + m.im, bi = p.im - m.im;
        if constexpr (EVEN) {
          ai += sg * (hp.im + hm.im);
          bi -= sg * (hp.im - hm.im);
        }
        ci = product<DATA_ROWS>(ai, t.c, ci);
        si = product<DATA_ROWS>(bi, t.s, si);
      }
    };
    load_trig(0, 0);
    if (AHEAD) load(0, 0);
#pragma unroll 1
    for (int d0 = 0; d0 < rounds; d0 += 2 * CH) {
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int dh = d0 + half * CH;
        if (dh + CH < rounds) {
          load_trig(1 - half, dh + CH);
          if (AHEAD) load(1 - half, dh + CH);
        }
        if (!AHEAD && dh < rounds) load(0, dh);
#pragma unroll
        for (int u = 0; u < CH; ++u) {
          if (dh + u < rounds) sum(dh + u, in[AHEAD ? half : 0][u], tr[half][u]);
        }
      }
    }
  }

  // Outputs q and n - q of accumulator element v.
  __device__ __forceinline__ void outputs(int v, Cd* o) const {
    if constexpr (REAL) {
      o[0] = Cd{cr[v], -sr[v]};
      o[1] = Cd{cr[v], sr[v]};
    } else {
      o[0] = Cd{cr[v] + si[v], ci[v] - sr[v]};
      o[1] = Cd{cr[v] - si[v], ci[v] + sr[v]};
    }
  }
};
// Tiles of 16 slots that hold the outputs q <= k: of even q (all of an odd
// length's), of odd q.
template <bool EVEN>
__device__ __forceinline__ int even_tiles(int k) {
  return (EVEN ? k / 2 : k) / kTile + 1;
}
template <bool EVEN>
__device__ __forceinline__ int odd_tiles(int k) {
  return EVEN ? ((k + 1) / 2 + kTile - 1) / kTile : 0;
}

// Hermitian fill of one pair of a line (reference symmetry_host.hpp:43-94): a
// non-zero lower entry (r < n / 2) wins, an upper one fills a zero lower one, the
// self-paired one is conjugated.
template <typename T>
__device__ __forceinline__ Pair<T> hermitian_pair(Pair<T> x, int n, int r) {
  if (2 * r == n) {
    x.p = cconj(x.p);
  } else if (r != 0) {
    if (cnonzero(x.p)) {
      x.m = cconj(x.p);
    } else if (cnonzero(x.m)) {
      x.p = cconj(x.m);
    }
  }
  return x;
}

// ------------------------------------------------------------- z kernels
//
// 16 sticks per workgroup; their values go through an LDS tile [stick][folded
// z], and the waves share out the output slots.

// Tile, then one element for repeated triplets.
template <typename T>
struct ZTile {
  Cx<T>* tile;  // [kDftSticks][pitch]
  int pitch, spare;
  __device__ ZTile(int n, int k) : pitch(z_pitch(n, k)) {
    tile = reinterpret_cast<Cx<T>*>(spfft_lds_dft);
    spare = kDftSticks * pitch;
  }
};
template <typename T>
size_t z_lds(int n, int k) {
  return (static_cast<size_t>(kDftSticks) * z_pitch(n, k) + 1) * sizeof(Cx<T>);
}

template <typename T, bool RC, bool EVEN>
__device__ __forceinline__ void z_backward_dft(const FastArgs<T>& a, int trigAt, int bid) {
  const int n = a.nz, kz = a.kz;
  const ZTile<T> z(n, kz);
  const int LZ = z.pitch, end = fold_end(n, kz);
  const int s0 = bid * kDftSticks;
  const int ns = min(kDftSticks, a.nst - s0);
  const Cx<T> zero = Cx<T>{T(0), T(0)};
  const Cx<T>* in = reinterpret_cast<const Cx<T>*>(a.in);
  const int s = threadIdx.x / kTile, l = threadIdx.x % kTile;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const Trig* tab = static_cast<const Trig*>(a.trig) + trigAt;
  using Sums = OutSums<T, EVEN, false, false, EVEN ? 1 : 2, false>;
  typename Sums::Roots head;
  int4 run = make_int4(0, 0, 0, 0);
  int e0 = 0, e1 = 0;
  if (a.hasRuns) {
    run = a.zInfo[min(s0 + s, a.nst - 1)];
  } else {
    e0 = a.stickBegin[s0];
    e1 = a.stickBegin[s0 + ns];
  }
  if (wave * kTile < out_slots(n)) head.first(n, kz, wave * kTile, tab);
  for (int t = threadIdx.x; t <= z.spare; t += kZWaves * kWave) z.tile[t] = zero;
  // the plane kernels read element nst of every row as zero
  if (bid == 0) {
    for (int t = threadIdx.x; t < n; t += kZWaves * kWave) {
      a.zbuf[static_cast<size_t>(t) * a.pitch + a.nst] = zero;
    }
  }
  lds_barrier();
  if (a.hasRuns) {
    // 16 lanes per stick, four values in flight each
    const int len = s < ns ? run.z : 0;
#pragma unroll 1
    for (int p0 = l; p0 < len; p0 += 4 * kTile) {
      Cx<T> x[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) x[u] = in[run.x + min(p0 + u * kTile, len - 1)];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        // lanes past the run's end write its last value again
        int zz = run.y + min(p0 + u * kTile, len - 1);
        zz -= zz >= n ? n : 0;
        z.tile[s * LZ + fold_at(n, kz, zz)] = x[u];
      }
    }
  } else {
#pragma unroll 1
    for (int e = e0 + static_cast<int>(threadIdx.x); e < e1; e += 4 * kZWaves * kWave) {
      int2 w[4];
      Cx<T> x[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = a.zEntries[min(e + u * kZWaves * kWave, e1 - 1)];
#pragma unroll
      for (int u = 0; u < 4; ++u) x[u] = in[w[u].x];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        // earlier copies of a repeated triplet go to the spare element; lanes
        // past the end write the last entry's value again
        z.tile[w[u].y < 0 ? z.spare : w[u].y] = x[u];
      }
    }
  }
  lds_barrier();
  const int line = lane % kTile;
  const Cx<T>* row = z.tile + line * LZ;
  const bool fill = RC && a.zeroZeroStick == 0 && s0 + line == 0;
  auto fetch = [&](int r) {
    Pair<T> x;
    x.p = row[r];
    x.m = row[end - r];
    if (RC && fill) x = hermitian_pair(x, n, r);
    return x;
  };
#pragma unroll 1
  for (int q0 = wave * kTile; q0 < out_slots(n); q0 += kZWaves * kTile) {
    if (q0 != wave * kTile) head.first(n, kz, q0, tab);
    Sums sums;
    sums.run(n, kz, q0, tab, head, fetch);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      Cd o[4];
      sums.outputs(n, q0, v, o);
      const int slot = q0 + tile_row(lane, v);
#pragma unroll
      for (int t = 0; t < (EVEN ? 4 : 2); ++t) {
        const int zz = out_index(n, slot, t);
        if (zz >= 0 && line < ns) {
          a.zbuf[static_cast<size_t>(zz) * a.pitch + s0 + line] = narrow<T>(o[t].re, o[t].im);
        }
      }
    }
  }
}

template <typename T, bool EVEN>
__device__ __forceinline__ void z_forward_dft(const FastArgs<T>& a, int trigAt, int bid) {
  const int n = a.nz, kz = a.kz;
  const ZTile<T> z(n, kz);
  const int LZ = z.pitch, end = fold_end(n, kz);
  const int s0 = bid * kDftSticks;
  const int ns = min(kDftSticks, a.nst - s0);
  const int s = threadIdx.x / kTile;
  int4 run = make_int4(0, 0, 0, 0);
  if (a.hasRuns) run = a.zInfo[min(s0 + s, a.nst - 1)];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int line = lane % kTile;
  // lines past the last stick read the last one; their results are not stored
  const Cx<T>* col = a.zbuf + s0 + min(line, ns - 1);
  auto fetch = [&](int r) {
    return quad_at<EVEN, T>(n, r, [&](int i) { return col[static_cast<size_t>(i) * a.pitch]; });
  };
  const Trig* tab = static_cast<const Trig*>(a.trig) + trigAt + out_table(n);
  const int even = even_tiles<EVEN>(kz), tiles = even + odd_tiles<EVEN>(kz);
#pragma unroll 1
  for (int tile = wave; tile < tiles; tile += kZWaves) {
    const int par = tile < even ? 0 : 1;
    const int j0 = (par ? tile - even : tile) * kTile;
    InSums<T, EVEN, false, false, EVEN ? 2 : 4, true> sums;
    sums.run(n, j0, par, tab, fetch);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int j = j0 + tile_row(lane, v);
      const int q = EVEN ? 2 * j + par : j;
      Cd o[2];
      sums.outputs(v, o);
      if (q <= kz) {
        z.tile[line * LZ + q] = narrow<T>(o[0].re, o[0].im);
        if (q != 0 && 2 * q != n) z.tile[line * LZ + end - q] = narrow<T>(o[1].re, o[1].im);
      }
    }
  }
  lds_barrier();
  Cx<T>* out = reinterpret_cast<Cx<T>*>(a.out);
  if (a.hasRuns) {
    const int len = s < ns ? run.z : 0;
    for (int pos = threadIdx.x % kTile; pos < len; pos += kTile) {
      int zz = run.y + pos;
      zz -= zz >= n ? n : 0;
      const Cx<T> c = z.tile[s * LZ + fold_at(n, kz, zz)];
      out[run.x + pos] = a.useScale ? cscale(c, a.scale) : c;
    }
  } else {
    const int e0 = a.stickBegin[s0], e1 = a.stickBegin[s0 + ns];
    for (int e = e0 + static_cast<int>(threadIdx.x); e < e1; e += kZWaves * kWave) {
      const int2 w = a.zEntries[e];
      const Cx<T> c = z.tile[w.y & 0x7fffffff];
      out[w.x] = a.useScale ? cscale(c, a.scale) : c;
    }
  }
}

// --------------------------------------------------------- plane kernels

// Launch constants of a plane kernel. A workgroup is (plane % 8, part, plane /
// 8 of its transform): workgroups are dealt to the 8 XCDs round robin, so the
// parts of a plane share one XCD's L2 for the plane's input.
struct PlaneArgs {
  int nx, ny, nz;
  int slotShift;     // log2 of the slots per workgroup
  int even;          // forward: parts of even output indices
  int blocks;        // plane blocks of a transform (batches)
  int trigX, trigY;  // the lengths' tables in FastArgs::trig
};

// Row pitch of the backward column tile: holds the folded y indices of the
// sticks (STAGED) and the rows, and is odd, so that the 16 columns of a tile
// row hit different banks.
__host__ __device__ constexpr int tile_pitch(int ny, int ky, int rows, bool staged) {
  const int in = staged ? fold_end(ny, ky) + 1 : 0;
  const int out = (rows + kTile - 1) / kTile * kTile;
  return (in > out ? in : out) | 1;
}

template <typename T>
__device__ __forceinline__ Trig trig_of(Tw<T> w) {
  if constexpr (sizeof(T) == 4) {
    return Trig{static_cast<double>(w.hi.re) + static_cast<double>(w.lo.re),
                -(static_cast<double>(w.hi.im) + static_cast<double>(w.lo.im))};
  } else {
    return Trig{w.re, -w.im};
  }
}
__device__ __forceinline__ Cd rotated(Cd acc, Cd x, Trig t) {  // acc + x exp(i t)
  return Cd{fma(x.re, t.c, fma(-x.im, t.s, acc.re)), fma(x.re, t.s, fma(x.im, t.c, acc.im))};
}
// Every stick's z sum at plane z into its tile cell: four lanes per stick, whose
// values are one run (FastArgs::zInfo).
template <typename T, bool RC>
__device__ __forceinline__ void sum_values(const FastArgs<T>& a, int n, int z, const Trig* tab,
                                           int P, Cx<T>* Y) {
  constexpr int L = 4, U = 4;
  const Cx<T>* in = reinterpret_cast<const Cx<T>*>(a.in);
  const int sub = threadIdx.x % L, step = blockDim.x / L;
  const int inc = L * z % n;
#pragma unroll 1
  for (int s = threadIdx.x / L; s < a.nst; s += step) {
    const int4 run = a.zInfo[s];
    const int cell = a.stickCell[s];
    Cd acc = Cd{0.0, 0.0};
    if (RC && s == 0 && a.zeroZeroStick == 0) {
      // the (0,0) stick is filled hermitian, pair by pair
      auto value = [&](int i) {
        int pos = i - run.y;
        pos += pos < 0 ? n : 0;
        return pos < run.z ? in[run.x + pos] : Cx<T>{T(0), T(0)};
      };
      for (int r = sub; r <= a.kz; r += L) {
        Pair<T> x;
        x.p = value(r);
        x.m = r != 0 && 2 * r != n ? value(n - r) : Cx<T>{T(0), T(0)};
        x = hermitian_pair(x, n, r);
        Trig t = tab[r * z % n];
        acc = rotated(acc, wide(x.p), t);
        t.s = -t.s;
        acc = rotated(acc, wide(x.m), t);
      }
    } else {
      int idx = (run.y + sub) * z % n;
#pragma unroll 1
      for (int p0 = sub; p0 < run.z; p0 += U * L) {
        Cx<T> x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = in[run.x + min(p0 + u * L, run.z - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (p0 + u * L < run.z) acc = rotated(acc, wide(x[u]), tab[idx]);
          idx += inc;
          idx -= idx >= n ? n : 0;
        }
      }
    }
#pragma unroll
    for (int d = 1; d < L; d *= 2) {
      acc.re += __shfl_xor(acc.re, d);
      acc.im += __shfl_xor(acc.im, d);
    }
    if (sub == 0) Y[(cell >> 16) * P + (cell & 0xffff)] = narrow<T>(acc.re, acc.im);
  }
}

// How the sticks of a plane reach the backward kernel: gathered from the [z]
// [stick] buffer through the [column][y] table (no room in LDS for more), from
// one pass over the plane's stick row into the tile as [column][folded y], or
// summed over z from the values themselves, with no z kernel before.
enum Source { kGather, kStaged, kValues };

// Backward: a workgroup owns the rows of its output slots of y. It computes
// those rows of every column, keeps them in LDS as [column][row], and transforms
// the rows. A wave's 16 columns are its own, so their rows overwrite their
// sticks.
template <typename T, bool RC, bool EX, bool EY, Source SRC>
__device__ __forceinline__ void xy_backward_dft(const FastArgs<T>& a, const PlaneArgs& p, int z,
                                                int part) {
  if (z >= a.nz) return;
  constexpr bool STAGED = SRC != kGather;
  const int nx = p.nx, ny = p.ny;
  constexpr int TY = EY ? 4 : 2, TX = EX ? 4 : 2;
  const int S = 1 << p.slotShift, rows = TY * S;
  const int q0 = part * S;
  const int kx = a.kx, ky = a.ky;
  const int P = tile_pitch(ny, ky, rows, STAGED);
  const int cols = tile_columns(nx, kx, RC);
  int* rowAt = reinterpret_cast<int*>(spfft_lds_dft);  // offset of a row in the plane, or -1
  Cx<T>* Y = reinterpret_cast<Cx<T>*>(rowAt + 4 * kTile);
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int threads = blockDim.x, waves = threads / kWave;
  const int line = lane % kTile;
  const Cx<T>* zrow = a.zbuf + static_cast<size_t>(z) * a.pitch;
  const Trig* trig = static_cast<const Trig*>(a.trig);
  if (threadIdx.x < 4 * kTile) {
    const int rl = threadIdx.x;
    const int y = rl < rows ? out_index(ny, q0 + (rl & (S - 1)), rl >> p.slotShift) : -1;
    rowAt[rl] = y < 0 ? -1 : y * nx;
  }
  using Sums = OutSums<T, EY, true, false, EY ? 1 : 2, !STAGED>;
  typename Sums::Roots head;
  head.first(ny, ky, q0, trig + p.trigY);  // every tile's: one tile of slots
  if constexpr (SRC == kValues) {
    const int nz = p.nz;
    Trig* tabZ = reinterpret_cast<Trig*>(Y + cols * P);
    for (int t = threadIdx.x; t < nz; t += threads) tabZ[t] = trig_of<T>(a.twZ[t]);
    for (int t = threadIdx.x; t < cols * P; t += threads) Y[t] = Cx<T>{T(0), T(0)};
    lds_barrier();
    sum_values<T, RC>(a, nz, z, tabZ, P, Y);
  } else if constexpr (STAGED) {
    // stickCell: tile column << 16 | folded y
    constexpr int U = 4;
    Cx<T> x[U];
    int cell[U];
    auto load = [&](int s0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int s = min(s0 + u * threads, a.nst - 1);
        cell[u] = a.stickCell[s];
        x[u] = at32(zrow, s);
      }
    };
    load(threadIdx.x);
    for (int t = threadIdx.x; t < cols * P; t += threads) Y[t] = Cx<T>{T(0), T(0)};
    lds_barrier();
#pragma unroll 1
    for (int s0 = threadIdx.x; s0 < a.nst; s0 += U * threads) {
      if (s0 != static_cast<int>(threadIdx.x)) load(s0);
      // lanes past the end write the last stick again
#pragma unroll
      for (int u = 0; u < U; ++u) Y[(cell[u] >> 16) * P + (cell[u] & 0xffff)] = x[u];
    }
  }
  lds_barrier();

  const int endY = fold_end(ny, ky);
#pragma unroll 1
  for (int i0 = wave * kTile; i0 < cols; i0 += waves * kTile) {
    const int i = i0 + line;
    // R2C: hermitian fill of the x = 0 column
    const bool fill = RC && i == 0;
    const int kmy = min(ky, (ny - 1) / 2);
    auto fetch = [&](int r) {
      Pair<T> v;
      if (STAGED) {
        v.p = Y[i * P + r];
        v.m = Y[i * P + endY - r];
      } else {
        const int* at = a.columnSticks + i * ny;
        const bool in = r <= ky, second = static_cast<unsigned>(r - 1) < static_cast<unsigned>(kmy);
        const int sp = at[in ? r : 0], sm = at[second ? ny - r : 0];
        v.p = at32(zrow, in ? sp : a.nst);
        v.m = at32(zrow, second ? sm : a.nst);
      }
      if (RC && fill) v = hermitian_pair(v, ny, r);
      return v;
    };
    Sums sums;
    sums.run(ny, ky, q0, trig + p.trigY, head, fetch);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      Cd o[4];
      sums.outputs(ny, q0, v, o);
      if (line < S) {
        Cx<T>* to = Y + (i0 + tile_row(lane, v)) * P + line;
#pragma unroll
        for (int t = 0; t < TY; ++t) to[t << p.slotShift] = narrow<T>(o[t].re, o[t].im);
      }
    }
  }
  const int rowTiles = (rows + kTile - 1) / kTile;
  const int items = rowTiles * ((out_slots(nx) + kTile - 1) / kTile);
  const int endX = fold_end(nx, kx);
  using RowSums = OutSums<T, EX, true, RC, EX ? 1 : 2, false>;
  typename RowSums::Roots rowHead;
  if (wave < items) rowHead.first(nx, kx, wave / rowTiles * kTile, trig + p.trigX);
  lds_barrier();

  // element type of the space domain
  using O = typename std::conditional<RC, T, Cx<T>>::type;
  O* plane = reinterpret_cast<O*>(a.out) + static_cast<size_t>(z) * ny * nx;
#pragma unroll 1
  for (int it = wave; it < items; it += waves) {
    const int r0 = (it % rowTiles) * kTile, xq0 = (it / rowTiles) * kTile;
    const Cx<T>* data = Y + r0 + line;
    auto fetch = [&](int r) {
      Pair<T> v;
      v.p = data[r * P];
      if (!RC) v.m = data[(endX - r) * P];
      return v;
    };
    if (it != wave) rowHead.first(nx, kx, xq0, trig + p.trigX);
    RowSums rowSums;
    rowSums.run(nx, kx, xq0, trig + p.trigX, rowHead, fetch);
    int xo[TX];
#pragma unroll
    for (int t = 0; t < TX; ++t) xo[t] = out_index(nx, xq0 + line, t);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int at = rowAt[r0 + tile_row(lane, v)];
      Cd o[4];
      rowSums.outputs(nx, xq0, v, o);
      if (at >= 0 && xo[0] >= 0) {
#pragma unroll
        for (int t = 0; t < TX; ++t) {
          if (t == 0 || xo[t] >= 0) {
            O value;
            if constexpr (RC) {
              value = static_cast<T>(o[t].re);
            } else {
              value = narrow<T>(o[t].re, o[t].im);
            }
            if (sizeof(T) == 8 && !RC && a.pastCache) {
              apart();
              store_stream(plane + at + xo[t], value);
              apart();
            } else {
              plane[at + xo[t]] = value;
            }
          }
        }
      }
    }
  }
}

// Forward: a workgroup owns the columns of its output slots of x. It computes
// those columns from every row of the plane, keeps them in LDS as [column][y],
// and transforms the columns.
template <typename T, bool RC, bool EX, bool EY>
__device__ __forceinline__ void xy_forward_dft(const FastArgs<T>& a, const PlaneArgs& p, int z,
                                               int part) {
  if (z >= a.nz) return;
  const int nx = p.nx, ny = p.ny;
  constexpr int TX = RC ? 1 : 2;  // columns per slot: q, and nx - q
  const int S = 1 << p.slotShift;
  const int par = EX && part >= p.even ? 1 : 0;
  const int j0 = (par ? part - p.even : part) * S;
  const int kx = a.kx, ky = a.ky;
  const int PY = ny | 1;
  const int ncolL = TX * S;  // columns of the workgroup
  Cx<T>* Y = reinterpret_cast<Cx<T>*>(spfft_lds_dft);
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int waves = blockDim.x / kWave;
  const int line = lane % kTile;
  const Trig* trig = static_cast<const Trig*>(a.trig);
  using I = typename std::conditional<RC, T, Cx<T>>::type;
  const I* plane = reinterpret_cast<const I*>(a.in) + static_cast<size_t>(z) * ny * nx;
#pragma unroll 1
  for (int y0 = wave * kTile; y0 < ny; y0 += waves * kTile) {
    const int row = min(y0 + line, ny - 1) * nx;
    auto fetch = [&](int r) {
      return quad_at<EX, T>(nx, r, [&](int i) {
        if constexpr (RC) {
          return Cx<T>{at32(plane, row + i), T(0)};
        } else {
          return at32(plane, row + i);
        }
      });
    };
    InSums<T, EX, false, RC, EX ? 1 : 2, true> sums;
    sums.run(nx, j0, par, trig + p.trigX + out_table(nx), fetch);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int j = tile_row(lane, v);
      Cd o[2];
      sums.outputs(v, o);
      if (j < S && y0 + line < ny) {
#pragma unroll
        for (int t = 0; t < TX; ++t) {
          Y[(t * S + j) * PY + y0 + line] = narrow<T>(o[t].re, o[t].im);
        }
      }
    }
  }
  lds_barrier();

  Cx<T>* zrow = a.zbuf + static_cast<size_t>(z) * a.pitch;
  const int colTiles = (ncolL + kTile - 1) / kTile;
  const int even = even_tiles<EY>(ky), tiles = even + odd_tiles<EY>(ky);
  const int endX = fold_end(nx, kx);
#pragma unroll 1
  for (int it = wave; it < colTiles * tiles; it += waves) {
    const int c0 = (it % colTiles) * kTile, yt = it / colTiles;
    const int yp = yt < even ? 0 : 1;
    const int yj0 = (yp ? yt - even : yt) * kTile;
    // sticks of this lane's outputs
    const int q = EY ? 2 * (yj0 + line) + yp : yj0 + line;
    int st[4][2];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      // column c = type * S + j: x of slot j's output, or nx minus it
      const int c = c0 + tile_row(lane, v);
      const int type = c >> p.slotShift, j = j0 + (c & (S - 1));
      const int qx = EX ? 2 * j + par : j;
      const bool ok = c < ncolL && q <= ky && qx <= kx &&
                      !(type == 1 && (qx == 0 || 2 * qx == nx));
      const int* at = a.columnSticks + (ok ? (type == 0 ? qx : endX - qx) * ny : 0);
      st[v][0] = at[ok ? q : 0];
      st[v][1] = at[ok && q != 0 ? ny - q : 0];
      if (!ok) st[v][0] = a.nst;
      if (!ok || q == 0 || 2 * q == ny) st[v][1] = a.nst;
    }
    const Cx<T>* data = Y + min(c0 + line, ncolL - 1) * PY;
    auto fetch = [&](int r) { return quad_at<EY, T>(ny, r, [&](int i) { return data[i]; }); };
    InSums<T, EY, true, false, EY ? 1 : 2, false> sums;
    sums.run(ny, yj0, yp, trig + p.trigY + out_table(ny), fetch);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      Cd o[2];
      sums.outputs(v, o);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if (st[v][t] < a.nst) zrow[st[v][t]] = narrow<T>(o[t].re, o[t].im);
      }
    }
  }
}

// ---- entry points: one transform (arguments by value) or a batch

template <typename T, bool RC, bool EVEN>
__global__ void __launch_bounds__(kZWaves * kWave)
    k_z_backward_dft(FastArgs<T> a, int trigAt) {
  z_backward_dft<T, RC, EVEN>(a, trigAt, blockIdx.x);
}
template <typename T, bool EVEN>
__global__ void __launch_bounds__(kZWaves * kWave) k_z_forward_dft(FastArgs<T> a, int trigAt) {
  z_forward_dft<T, EVEN>(a, trigAt, blockIdx.x);
}
template <typename T, bool RC, bool EVEN>
__global__ void __launch_bounds__(kZWaves * kWave)
    k_z_backward_dft_batch(const FastArgs<T>* __restrict__ batch, const int2* __restrict__ map,
                           int useRuns, int trigAt) {
  const int2 m = map[blockIdx.x];
  FastArgs<T> a = on_global(batch[m.x], batch);
  a.hasRuns = a.hasRuns && useRuns;
  z_backward_dft<T, RC, EVEN>(a, trigAt, m.y);
}
template <typename T, bool EVEN>
__global__ void __launch_bounds__(kZWaves * kWave)
    k_z_forward_dft_batch(const FastArgs<T>* __restrict__ batch, const int2* __restrict__ map,
                          int useRuns, int trigAt) {
  const int2 m = map[blockIdx.x];
  FastArgs<T> a = on_global(batch[m.x], batch);
  a.hasRuns = a.hasRuns && useRuns;
  z_forward_dft<T, EVEN>(a, trigAt, m.y);
}
// SRC: backward only
template <typename T, bool FWD, bool RC, bool EX, bool EY, Source SRC>
__device__ __forceinline__ void xy_dft(const FastArgs<T>& a, const PlaneArgs& p, int block) {
  const int z = a.zBegin + 8 * block + static_cast<int>(blockIdx.x);
  if constexpr (FWD) {
    xy_forward_dft<T, RC, EX, EY>(a, p, z, blockIdx.y);
  } else {
    xy_backward_dft<T, RC, EX, EY, SRC>(a, p, z, blockIdx.y);
  }
}
// Waves per SIMD: two workgroups of eight waves share a CU where the kernel's
// accumulators leave room for it without spills.
template <bool FWD, bool EX, bool EY>
constexpr int plane_waves() {
  return !FWD && (EX || EY) ? 3 : 4;
}
template <typename T, bool FWD, bool RC, bool EX, bool EY, Source SRC>
__global__ void __launch_bounds__(kMaxWaves * kWave) __attribute__((amdgpu_waves_per_eu(plane_waves<FWD, EX, EY>())))
    k_xy_dft(FastArgs<T> a, PlaneArgs p) {
  xy_dft<T, FWD, RC, EX, EY, SRC>(a, p, blockIdx.z);
}
template <typename T, bool FWD, bool RC, bool EX, bool EY, Source SRC>
__global__ void __launch_bounds__(kMaxWaves * kWave) __attribute__((amdgpu_waves_per_eu(plane_waves<FWD, EX, EY>())))
    k_xy_dft_batch(const FastArgs<T>* __restrict__ batch, PlaneArgs p) {
  const int t = blockIdx.z / p.blocks;
  xy_dft<T, FWD, RC, EX, EY, SRC>(on_global(batch[t], batch), p, blockIdx.z - t * p.blocks);
}

// Raise the dynamic LDS limit of a kernel once per process.
template <typename Kernel>
void prepare_lds(Kernel kernel, size_t lds) {
  if (lds > kLdsMax) throw GPUFFTError();
  if (lds <= kLdsDefault) return;
  static std::mutex mutex;
  static std::unordered_map<const void*, bool> raised;
  const void* key = reinterpret_cast<const void*>(kernel);
  std::lock_guard<std::mutex> lock(mutex);
  if (raised.count(key)) return;
  check_hip(hipFuncSetAttribute(key, hipFuncAttributeMaxDynamicSharedMemorySize,
                                static_cast<int>(kLdsMax)));
  raised[key] = true;
}

template <typename Kernel, typename... Args>
void launch(Kernel kernel, const char* name, dim3 grid, int threads, size_t lds,
            hipStream_t stream, Args... args) {
  prepare_lds(kernel, lds);
  prof::KernelSpan span(stream, name, true);
  hipExtLaunchKernelGGL(kernel, grid, dim3(threads), lds, stream, span.start(), span.stop(), 0,
                        args...);
  check_launch();
}

// Workgroups per plane, slots (rows or columns by type) per workgroup and LDS
// bytes of one launch of the plane kernels.
struct Plan {
  int parts = 0;        // workgroups per plane
  int slotShift = 0;    // log2 of the slots per workgroup
  int even = 0;         // forward: workgroups of even output indices (even lengths)
  int waves = 4;        // per workgroup
  Source source = kGather;  // backward
  size_t lds = 0;
};

// `planes`: planes of the launch (all transforms of a batch); kx, ky: widest of
// it. A part costs a whole tile of 16 slots in its first transform however few
// it owns, so a plane is cut into fewer slots per part only while the launch
// leaves most CUs idle or the tile does not fit in LDS, and never below one tile
// of 16 rows (columns). nz > 0: backward from the values.
template <typename T>
Plan plane_plan(bool forward, bool r2c, int nx, int ny, int kx, int ky, int planes, int nz = 0) {
  constexpr int kEnough = 160;  // workgroups, of 256 CUs
  Plan plan;
  const bool evenX = nx % 2 == 0;
  const int total = forward ? (evenX ? kx / 2 + 1 : kx + 1) : out_slots(ny);
  const int types = forward ? (r2c ? 1 : 2) : out_types(ny);
  for (plan.slotShift = 4;; --plan.slotShift) {
    const int slots = 1 << plan.slotShift, lines = types * slots;
    if (forward) {
      plan.even = evenX ? (kx / 2 + slots) / slots : 0;
      plan.parts = evenX ? plan.even + ((kx + 1) / 2 + slots - 1) / slots : (kx + slots) / slots;
      plan.lds = static_cast<size_t>(lines) * (ny | 1) * sizeof(Cx<T>);
    } else {
      plan.parts = (total + slots - 1) / slots;
      auto bytes = [&](bool staged) {
        return 4 * kTile * sizeof(int) + static_cast<size_t>(tile_columns(nx, kx, r2c)) *
                                             tile_pitch(ny, ky, lines, staged) * sizeof(Cx<T>);
      };
      plan.source = bytes(true) <= kLdsMax ? kStaged : kGather;
      if (nz > 0) plan.source = kValues;
      plan.lds = bytes(plan.source != kGather) + nz * sizeof(Trig);
    }
    if (lines <= kTile) break;
    if (plan.lds <= kLdsMax && planes * plan.parts >= kEnough && slots / 2 < total) break;
  }
  // a wave per tile of the larger transform
  const int lines = types << plan.slotShift;
  auto tiles = [](int n) { return (n + kTile - 1) / kTile; };
  const int work = forward ? std::max(tiles(ny), tiles(lines) * (tiles(ky + 1)))
                           : std::max(tile_columns(nx, kx, r2c) / kTile,
                                      tiles(lines) * tiles(out_slots(nx)));
  // (and all of them for the sums over z)
  plan.waves = work > 4 || plan.source == kValues ? kMaxWaves : 4;
  return plan;
}

// f(kernel) with the plane kernel for the run-time choices.
template <typename T, bool BATCH, bool FWD, bool RC, Source SRC, typename F>
void plane_kernel(bool evenX, bool evenY, F&& f) {
#define SPFFT_PLANE_CASE(EX, EY)                          \
  if (evenX == EX && evenY == EY) {                       \
    if constexpr (BATCH) {                                \
      return f(k_xy_dft_batch<T, FWD, RC, EX, EY, SRC>);  \
    } else {                                              \
      return f(k_xy_dft<T, FWD, RC, EX, EY, SRC>);        \
    }                                                     \
  }
  SPFFT_PLANE_CASE(true, true)
  SPFFT_PLANE_CASE(true, false)
  SPFFT_PLANE_CASE(false, true)
  SPFFT_PLANE_CASE(false, false)
#undef SPFFT_PLANE_CASE
}
template <typename T, bool BATCH, bool RC, typename F>
void plane_kernel(bool forward, bool evenX, bool evenY, Source source, F&& f) {
  if (forward) {
    plane_kernel<T, BATCH, true, RC, kGather>(evenX, evenY, f);
  } else if (source == kGather) {
    plane_kernel<T, BATCH, false, RC, kGather>(evenX, evenY, f);
  } else if (source == kStaged) {
    plane_kernel<T, BATCH, false, RC, kStaged>(evenX, evenY, f);
  } else {
    plane_kernel<T, BATCH, false, RC, kValues>(evenX, evenY, f);
  }
}
template <typename T, bool BATCH, typename F>
void plane_kernel(bool forward, bool r2c, bool evenX, bool evenY, Source source, F&& f) {
  r2c ? plane_kernel<T, BATCH, true>(forward, evenX, evenY, source, f)
      : plane_kernel<T, BATCH, false>(forward, evenX, evenY, source, f);
}

PlaneArgs plane_args(const Plan& plan, const DftTables& t, int nx, int ny, int nz, int blocks) {
  return PlaneArgs{nx, ny, nz, plan.slotShift, plan.even, blocks, t.at[0], t.at[1]};
}

}  // namespace

template <typename T>
bool dft_plane_supported(bool r2c, int nx, int ny, int kx, int ky) {
  if (nx > kDftMaxLength || ny > kDftMaxLength) return false;
  // one plane: the smallest parts
  return plane_plan<T>(false, r2c, nx, ny, kx, ky, 1).lds <= kLdsMax &&
         plane_plan<T>(true, r2c, nx, ny, kx, ky, 1).lds <= kLdsMax;
}

template <typename T>
bool dft_values_supported(bool r2c, int nx, int ny, int nz, int kx, int ky) {
  // any planes: the largest tile is the one of most slots
  return dft_plane_supported<T>(r2c, nx, ny, kx, ky) &&
         plane_plan<T>(false, r2c, nx, ny, kx, ky, 1 << 20, nz).lds <= kLdsMax;
}

template <typename T>
void launch_dft_xy(bool forward, int nx, int ny, int fromValues, const FastArgs<T>& a,
                   hipStream_t stream) {
  const bool rc = a.r2c != 0;
  const int planes = a.nz - a.zBegin;
  const Plan plan = plane_plan<T>(forward, rc, nx, ny, a.kx, a.ky, planes, fromValues);
  const int blocks = (planes + 7) / 8;
  const PlaneArgs p = plane_args(plan, DftTables(nx, ny, 1), nx, ny, fromValues, blocks);
  plane_kernel<T, false>(forward, rc, nx % 2 == 0, ny % 2 == 0, plan.source, [&](auto kernel) {
    launch(kernel, forward ? "k_xy_forward_dft" : "k_xy_backward_dft",
           dim3(8, plan.parts, blocks), plan.waves * kWave, plan.lds, stream, a, p);
  });
}

template <typename T>
void launch_dft_xy_batch(bool forward, bool r2c, int nx, int ny, int fromValues, int kx, int ky,
                         const FastArgs<T>* batch, int ntrans, int nz, hipStream_t stream) {
  const Plan plan = plane_plan<T>(forward, r2c, nx, ny, kx, ky, nz * ntrans, fromValues);
  const int blocks = (nz + 7) / 8;
  const PlaneArgs p = plane_args(plan, DftTables(nx, ny, 1), nx, ny, fromValues, blocks);
  plane_kernel<T, true>(forward, r2c, nx % 2 == 0, ny % 2 == 0, plan.source, [&](auto kernel) {
    launch(kernel, forward ? "k_xy_forward_dft_batch" : "k_xy_backward_dft_batch",
           dim3(8, plan.parts, blocks * ntrans), plan.waves * kWave, plan.lds, stream, batch, p);
  });
}

template <typename T>
void launch_dft_z(bool forward, int nx, int ny, const FastArgs<T>& a, hipStream_t stream) {
  const int blocks = (a.nst + kDftSticks - 1) / kDftSticks;
  const bool even = a.nz % 2 == 0;
  auto kernel =
      forward ? (even ? k_z_forward_dft<T, true> : k_z_forward_dft<T, false>)
      : a.r2c ? (even ? k_z_backward_dft<T, true, true> : k_z_backward_dft<T, true, false>)
              : (even ? k_z_backward_dft<T, false, true> : k_z_backward_dft<T, false, false>);
  launch(kernel, forward ? "k_z_forward_dft" : "k_z_backward_dft", dim3(blocks),
         kZWaves * kWave, z_lds<T>(a.nz, a.kz), stream, a, DftTables(nx, ny, a.nz).at[2]);
}

template <typename T>
void launch_dft_z_batch(bool forward, bool r2c, int nx, int ny, int nz, int kz,
                        const FastArgs<T>* batch, const int2* map, int blocks, bool useRuns,
                        hipStream_t stream) {
  const bool even = nz % 2 == 0;
  auto kernel = forward ? (even ? k_z_forward_dft_batch<T, true> : k_z_forward_dft_batch<T, false>)
                : r2c   ? (even ? k_z_backward_dft_batch<T, true, true>
                                : k_z_backward_dft_batch<T, true, false>)
                        : (even ? k_z_backward_dft_batch<T, false, true>
                                : k_z_backward_dft_batch<T, false, false>);
  launch(kernel, forward ? "k_z_forward_dft_batch" : "k_z_backward_dft_batch", dim3(blocks),
         kZWaves * kWave, z_lds<T>(nz, kz), stream, batch, map, useRuns ? 1 : 0,
         DftTables(nx, ny, nz).at[2]);
}

#define SPFFT_INSTANTIATE_DFT(T)                                                              \
  template bool dft_plane_supported<T>(bool, int, int, int, int);                             \
  template bool dft_values_supported<T>(bool, int, int, int, int, int);                       \
  template void launch_dft_xy<T>(bool, int, int, int, const FastArgs<T>&, hipStream_t);       \
  template void launch_dft_xy_batch<T>(bool, bool, int, int, int, int, int,                   \
                                       const FastArgs<T>*, int, int, hipStream_t);            \
  template void launch_dft_z<T>(bool, int, int, const FastArgs<T>&, hipStream_t);             \
  template void launch_dft_z_batch<T>(bool, bool, int, int, int, int, const FastArgs<T>*,     \
                                      const int2*, int, bool, hipStream_t);

// One precision per translation unit: dft_kernels_float.hip includes this file
// with SPFFT_DFT_FLOAT set.
#ifdef SPFFT_DFT_FLOAT
SPFFT_INSTANTIATE_DFT(float)
#else
SPFFT_INSTANTIATE_DFT(double)


void build_dft_tables(void* tables, int nx, int ny, int nz, hipStream_t stream) {
  const DftTables at(nx, ny, nz);
  const int n[3] = {nx, ny, nz};
  for (int d = 0; d < 3; ++d) {
    if ((d > 0 && n[d] == nx) || (d == 2 && n[d] == ny)) continue;  // shared
    const int count = out_table(n[d]) + in_table(n[d]);
    hipLaunchKernelGGL(k_dft_trig, dim3((count + 255) / 256), dim3(256), 0, stream,
                       static_cast<Trig*>(tables) + at.at[d], n[d]);
    check_launch();
  }
}
#endif

}  // namespace spfft

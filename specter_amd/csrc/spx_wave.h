// Line FFTs with compile-time plans, one wavefront or a part of one per line
// (gfx950, wave64).
//
// The general engine (spx_engine.h) reads its radix sequence from the plan at
// run time and spreads long lines over several wavefronts, which costs index
// arithmetic per butterfly, scalar registers and a workgroup barrier per pass.
// Here the length M of the FFT and its radices are fixed at compile time:
// every pass knows M, its radix R and its stride Ns, so the index arithmetic
// folds into constants and immediate LDS offsets, and L <= 64 lanes of one
// wavefront own one line, so the passes synchronise with the wavefront's own
// ordering of its LDS accesses (no s_barrier).  Each lane runs ceil(M/R/L)
// butterflies of a pass; they are loaded, transformed and stored together, in
// place.  Composite radices (6 ... 45) run as two-level DFTs in registers with
// their inner twiddles as constants, so a plan needs fewer LDS passes.
// The DFT length n of a Bluestein plan is a run-time value (2n - 1 <= M): a
// ladder of M serves every length.
//
// Conventions are the engine's: forward transforms, the same Bluestein
// factorisation (chirp, FFT, filter, FFT, chirp), so a plan and the engine
// agree to rounding.
#pragma once

#include "spx_engine.h"

namespace spx {

// A wavefront's LDS instructions complete in order: between the passes of a
// line owned by one wavefront only the compiler has to be kept from moving
// accesses across the pass boundary.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// cos(2 pi k / R) and sin(2 pi k / R), k < R, for the composite radices
// (computed in 50-digit decimal arithmetic, printed to 24 digits).
template <int R>
struct RootTab;
template <>
struct RootTab<6> {
  static constexpr double c[6] = {
      1.000000000000000000000000, 0.500000000000000000000000, -0.500000000000000000000000,
      -1.000000000000000000000000, -0.500000000000000000000000, 0.500000000000000000000000};
  static constexpr double s[6] = {
      0.0, 0.866025403784438646763723, 0.866025403784438646763723,
      0.0, -0.866025403784438646763723, -0.866025403784438646763723};
};
template <>
struct RootTab<9> {
  static constexpr double c[9] = {
      1.000000000000000000000000, 0.766044443118978035202393, 0.173648177666930348851717,
      -0.500000000000000000000000, -0.939692620785908384054109, -0.939692620785908384054109,
      -0.500000000000000000000000, 0.173648177666930348851717, 0.766044443118978035202393};
  static constexpr double s[9] = {
      0.0, 0.642787609686539326322643, 0.984807753012208059366743,
      0.866025403784438646763723, 0.342020143325668733044100, -0.342020143325668733044100,
      -0.866025403784438646763723, -0.984807753012208059366743, -0.642787609686539326322643};
};
template <>
struct RootTab<10> {
  static constexpr double c[10] = {
      1.000000000000000000000000, 0.809016994374947424102293, 0.309016994374947424102293,
      -0.309016994374947424102293, -0.809016994374947424102293, -1.000000000000000000000000,
      -0.809016994374947424102293, -0.309016994374947424102293, 0.309016994374947424102293,
      0.809016994374947424102293};
  static constexpr double s[10] = {
      0.0, 0.587785252292473129168706, 0.951056516295153572116439,
      0.951056516295153572116439, 0.587785252292473129168706, 0.0,
      -0.587785252292473129168706, -0.951056516295153572116439, -0.951056516295153572116439,
      -0.587785252292473129168706};
};
template <>
struct RootTab<12> {
  static constexpr double c[12] = {
      1.000000000000000000000000, 0.866025403784438646763723, 0.500000000000000000000000,
      0.0, -0.500000000000000000000000, -0.866025403784438646763723,
      -1.000000000000000000000000, -0.866025403784438646763723, -0.500000000000000000000000,
      0.0, 0.500000000000000000000000, 0.866025403784438646763723};
  static constexpr double s[12] = {
      0.0, 0.500000000000000000000000, 0.866025403784438646763723,
      1.000000000000000000000000, 0.866025403784438646763723, 0.500000000000000000000000,
      0.0, -0.500000000000000000000000, -0.866025403784438646763723,
      -1.000000000000000000000000, -0.866025403784438646763723, -0.500000000000000000000000};
};
template <>
struct RootTab<15> {
  static constexpr double c[15] = {
      1.000000000000000000000000, 0.913545457642600895502128, 0.669130606358858213826273,
      0.309016994374947424102293, -0.104528463267653471399834, -0.500000000000000000000000,
      -0.809016994374947424102293, -0.978147600733805637928567, -0.978147600733805637928567,
      -0.809016994374947424102293, -0.500000000000000000000000, -0.104528463267653471399834,
      0.309016994374947424102293, 0.669130606358858213826273, 0.913545457642600895502128};
  static constexpr double s[15] = {
      0.0, 0.406736643075800207753986, 0.743144825477394235014697,
      0.951056516295153572116439, 0.994521895368273336922692, 0.866025403784438646763723,
      0.587785252292473129168706, 0.207911690817759337101742, -0.207911690817759337101742,
      -0.587785252292473129168706, -0.866025403784438646763723, -0.994521895368273336922692,
      -0.951056516295153572116439, -0.743144825477394235014697, -0.406736643075800207753986};
};
template <>
struct RootTab<16> {
  static constexpr double c[16] = {
      1.000000000000000000000000, 0.923879532511286756128183, 0.707106781186547524400844,
      0.382683432365089771728460, 0.0, -0.382683432365089771728460,
      -0.707106781186547524400844, -0.923879532511286756128183, -1.000000000000000000000000,
      -0.923879532511286756128183, -0.707106781186547524400844, -0.382683432365089771728460,
      0.0, 0.382683432365089771728460, 0.707106781186547524400844,
      0.923879532511286756128183};
  static constexpr double s[16] = {
      0.0, 0.382683432365089771728460, 0.707106781186547524400844,
      0.923879532511286756128183, 1.000000000000000000000000, 0.923879532511286756128183,
      0.707106781186547524400844, 0.382683432365089771728460, 0.0,
      -0.382683432365089771728460, -0.707106781186547524400844, -0.923879532511286756128183,
      -1.000000000000000000000000, -0.923879532511286756128183, -0.707106781186547524400844,
      -0.382683432365089771728460};
};
template <>
struct RootTab<18> {
  static constexpr double c[18] = {
      1.000000000000000000000000, 0.939692620785908384054109, 0.766044443118978035202393,
      0.500000000000000000000000, 0.173648177666930348851717, -0.173648177666930348851717,
      -0.500000000000000000000000, -0.766044443118978035202393, -0.939692620785908384054109,
      -1.000000000000000000000000, -0.939692620785908384054109, -0.766044443118978035202393,
      -0.500000000000000000000000, -0.173648177666930348851717, 0.173648177666930348851717,
      0.500000000000000000000000, 0.766044443118978035202393, 0.939692620785908384054109};
  static constexpr double s[18] = {
      0.0, 0.342020143325668733044100, 0.642787609686539326322643,
      0.866025403784438646763723, 0.984807753012208059366743, 0.984807753012208059366743,
      0.866025403784438646763723, 0.642787609686539326322643, 0.342020143325668733044100,
      0.0, -0.342020143325668733044100, -0.642787609686539326322643,
      -0.866025403784438646763723, -0.984807753012208059366743, -0.984807753012208059366743,
      -0.866025403784438646763723, -0.642787609686539326322643, -0.342020143325668733044100};
};
template <>
struct RootTab<20> {
  static constexpr double c[20] = {
      1.000000000000000000000000, 0.951056516295153572116439, 0.809016994374947424102293,
      0.587785252292473129168706, 0.309016994374947424102293, 0.0,
      -0.309016994374947424102293, -0.587785252292473129168706, -0.809016994374947424102293,
      -0.951056516295153572116439, -1.000000000000000000000000, -0.951056516295153572116439,
      -0.809016994374947424102293, -0.587785252292473129168706, -0.309016994374947424102293,
      0.0, 0.309016994374947424102293, 0.587785252292473129168706,
      0.809016994374947424102293, 0.951056516295153572116439};
  static constexpr double s[20] = {
      0.0, 0.309016994374947424102293, 0.587785252292473129168706,
      0.809016994374947424102293, 0.951056516295153572116439, 1.000000000000000000000000,
      0.951056516295153572116439, 0.809016994374947424102293, 0.587785252292473129168706,
      0.309016994374947424102293, 0.0, -0.309016994374947424102293,
      -0.587785252292473129168706, -0.809016994374947424102293, -0.951056516295153572116439,
      -1.000000000000000000000000, -0.951056516295153572116439, -0.809016994374947424102293,
      -0.587785252292473129168706, -0.309016994374947424102293};
};

// v * exp(-2 pi i k / R); k is a constant after unrolling, so the table
// entries become immediates.  Exact for multiples of pi/2.
template <typename T, int R>
__device__ __forceinline__ cpx<T> wroot(cpx<T> v, int k) {
  k %= R;
  if (k == 0) return v;
  if ((4 * k) % R == 0) {
    const int q = 4 * k / R;
    if (q == 1) return mkc<T>(v.y, -v.x);
    if (q == 2) return mkc<T>(-v.x, -v.y);
    return mkc<T>(-v.y, v.x);
  }
  return cmul(v, mkc<T>(T(RootTab<R>::c[k]), T(-RootTab<R>::s[k])));
}

template <typename T, int R>
struct WDft;

// R = P Q as P-point DFTs over n1 of x[Q n1 + n2], twiddles W_R^(n2 k1),
// Q-point DFTs over n2, output X[k1 + P k2].
template <typename T, int P, int Q>
struct DftPQ {
  static __device__ __forceinline__ void run(cpx<T>* v) {
    constexpr int R = P * Q;
    cpx<T> a[Q][P];
#pragma unroll
    for (int n2 = 0; n2 < Q; ++n2) {
      cpx<T> t[P];
#pragma unroll
      for (int n1 = 0; n1 < P; ++n1) t[n1] = v[Q * n1 + n2];
      WDft<T, P>::run(t);
#pragma unroll
      for (int k1 = 0; k1 < P; ++k1) a[n2][k1] = wroot<T, R>(t[k1], n2 * k1);
    }
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) {
      cpx<T> t[Q];
#pragma unroll
      for (int n2 = 0; n2 < Q; ++n2) t[n2] = a[n2][k1];
      WDft<T, Q>::run(t);
#pragma unroll
      for (int k2 = 0; k2 < Q; ++k2) v[k1 + P * k2] = t[k2];
    }
  }
};

// Radix-R DFT in registers with constant roots: the engine's butterflies for
// 2, 3, 4, 5, 7, 8, 11, 13 (their roots are immediates), two-level otherwise.
template <typename T, int R>
struct WDft {
  static __device__ __forceinline__ void run(cpx<T>* v) { Dft<T, R>::run(v, nullptr, 0); }
};
template <typename T>
struct WDft<T, 6> : DftPQ<T, 2, 3> {};
template <typename T>
struct WDft<T, 9> : DftPQ<T, 3, 3> {};
template <typename T>
struct WDft<T, 10> : DftPQ<T, 2, 5> {};
template <typename T>
struct WDft<T, 12> : DftPQ<T, 4, 3> {};
template <typename T>
struct WDft<T, 15> : DftPQ<T, 3, 5> {};
template <typename T>
struct WDft<T, 16> : DftPQ<T, 4, 4> {};
template <typename T>
struct WDft<T, 18> : DftPQ<T, 2, 9> {};
template <typename T>
struct WDft<T, 20> : DftPQ<T, 4, 5> {};

constexpr int ceil_sqrt(int r) {
  int q = 1;
  while (q * q < r) ++q;
  return q;
}

// Stage twiddles of a pass of radix R at stride Ns, v[r] *= W_(Ns R)^(r jm).
// The plan's table holds each pass's factors in the order its lanes read them,
// W_(Ns R)^(r jm) at r Ns + jm - 1 (the passes fill M - 1 entries without
// gaps): neighbouring lanes read neighbouring entries, where reads of one
// M-entry table of W_M at r jm M/(Ns R) met on few LDS banks (the dual y pass of
// 256-point lines 307 us instead of 248, of 512-point lines 2.57 ms instead of
// 2.25).  TWM 0: every factor read from the table.  TWM 2: those of r = a < q
// and r = q b, q = ceil(sqrt(R)), are read and the others formed as products.  Direct lines are bound by memory
// either way and take TWM 0, the engine's accuracy; Bluestein lines, whose
// error the chirp convolution sets, are 4-14 % faster with fewer reads.
template <typename T, int R, int TWM, int Ns>
__device__ __forceinline__ void stage_twiddle(cpx<T>* v, const cpx<T>* tw, int jm) {
  const cpx<T>* const t = tw + (jm - 1);
  if constexpr (TWM == 0 || R <= 4) {
#pragma unroll
    for (int r = 1; r < R; ++r) v[r] = cmul(v[r], t[r * Ns]);
  } else {
    constexpr int q = ceil_sqrt(R), nb = (R + q - 1) / q;
    cpx<T> wa[q], wb[nb];
#pragma unroll
    for (int a = 1; a < q; ++a) wa[a] = t[a * Ns];
#pragma unroll
    for (int b = 1; b < nb; ++b) wb[b] = t[b * q * Ns];
#pragma unroll
    for (int r = 1; r < R; ++r) {
      const int a = r % q, b = r / q;
      v[r] = cmul(v[r], b == 0 ? wa[a] : (a == 0 ? wb[b] : cmul(wb[b], wa[a])));
    }
  }
}

// A padded plan keeps the line with one slot of padding per R1 elements
// between its first two passes: the first stores element j R1 + r, and R1
// slots of 8 or 16 bytes between neighbouring lanes fall on few banks when R1
// is a multiple of 4.  The second pass reads j + r M/R2, whose padded place is
// a run-time part of j plus a constant of r.
// One in-place Stockham pass of radix R at stride Ns on the M-point line x
// (LDS), L lanes, twiddle table tw (M entries).  LD / ST: chirp or Rader gather
// on load; filter, chirp or Rader scatter on store (the filter and chirp
// tables hold M entries).  Rader: t.x0 is the line's element 0, X0 its output 0,
// kept by the lane that stores element 0 of the first FFT.
// PADIN: the input is padded per PADIN elements (0: not); PADOUT: this first
// pass leaves its output padded.
template <typename T>
struct WaveTab {
  const cpx<T>* __restrict__ filt;
  const cpx<T>* __restrict__ chirp;
  const int* __restrict__ gin;
  const int* __restrict__ gout;
  cpx<T> x0, X0;
};

template <typename T, int M, int L, int Ns, int R, int NMAX, int LD, int ST, int TWM, int PADIN,
          int PADOUT>
__device__ __forceinline__ void wave_pass(cpx<T>* x, int lane, const cpx<T>* tw, int n,
                                          WaveTab<T>& t) {
  constexpr int nb = M / R;
  constexpr int NR = (nb + L - 1) / L;
  static_assert(M % R == 0, "radix does not divide the length");
  static_assert(PADIN == 0 || nb % PADIN == 0, "padded input needs whole rows");
  // the filter and chirp factors are loaded before the line is synchronised,
  // behind the butterflies; lines of 14 and more points per lane have no
  // registers to spare for that (spills) and load them with the stores
  constexpr bool LATE = M / L >= 14;
  auto apply = [&](cpx<T>* u, int base) {
    if constexpr (ST == ST_FILTER) {
      if (base == 0) t.X0 = cadd(t.x0, u[0]);
#pragma unroll
      for (int r = 0; r < R; ++r) u[r] = cconj(cmul(u[r], t.filt[base + r * Ns]));
    } else if constexpr (ST == ST_CHIRP) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (r * Ns < NMAX) u[r] = cmul(cconj(u[r]), t.chirp[base + r * Ns]);
    }
  };
  // butterflies of this pass, opaque to the compiler for TWM 0: rounds it cannot
  // merge into one block contract their products as the general engine's do
  // (line_pass), so these plans return the engine's bits (a few percent of the y
  // and x passes of 256 points in float64 against constant bounds)
  int count = nb;
  if constexpr (TWM == 0) asm volatile("" : "+s"(count));
  cpx<T> v[NR][R];
#pragma unroll
  for (int b = 0; b < NR; ++b) {
    const unsigned j = unsigned(lane) + unsigned(L * b);
    if ((TWM != 0 && (b + 1) * L <= nb) || j < unsigned(count)) {
      const int jm = Ns > 1 ? int(j % unsigned(Ns)) : 0;
      if constexpr (LD == LD_CHIRP) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          if (r * nb >= NMAX) {
            v[b][r] = mkc<T>(0, 0);
          } else {
            const int q = int(j) + r * nb;
            const cpx<T> u = cmul(x[q], t.chirp[q]);
            v[b][r] = q < n ? u : mkc<T>(0, 0);
          }
        }
      } else if constexpr (LD == LD_GATHER) {
#pragma unroll
        for (int r = 0; r < R; ++r) v[b][r] = x[t.gin[int(j) + r * nb]];
      } else if constexpr (PADIN > 0) {
        const int o = int(j) + int(j / unsigned(PADIN));
#pragma unroll
        for (int r = 0; r < R; ++r) v[b][r] = x[o + r * (nb / PADIN) * (PADIN + 1)];
      } else {
#pragma unroll
        for (int r = 0; r < R; ++r) v[b][r] = x[int(j) + r * nb];
      }
      if constexpr (Ns > 1) stage_twiddle<T, R, TWM, Ns>(v[b], tw, jm);
      // TWM 0 runs the engine's butterflies, radix 9 with its roots from the table
      if constexpr (TWM == 0 && R == 9) Dft<T, 9>::run(v[b], tw + M, 1);
      else WDft<T, R>::run(v[b]);
      if constexpr (!LATE) apply(v[b], (int(j) - jm) * R + jm);
    }
  }
  wave_sync();
#pragma unroll
  for (int b = 0; b < NR; ++b) {
    const unsigned j = unsigned(lane) + unsigned(L * b);
    if ((TWM != 0 && (b + 1) * L <= nb) || j < unsigned(count)) {
      const int jm = Ns > 1 ? int(j % unsigned(Ns)) : 0;
      const int base = PADOUT ? int(j) * (R + 1) : (int(j) - jm) * R + jm;
      if constexpr (LATE) apply(v[b], base);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if constexpr (ST == ST_CHIRP) {
          if (r * Ns < NMAX && base + r * Ns < n) x[base + r * Ns] = v[b][r];
        } else if constexpr (ST == ST_SCATTER) {
          x[t.gout[base + r * Ns]] = cadd(t.x0, cconj(v[b][r]));
        } else {
          x[base + r * Ns] = v[b][r];
        }
      }
    }
  }
  wave_sync();
}

// The passes of one M-point FFT: the first loads with LD, the last stores
// with ST.
template <typename T, int M, int L, int Ns, int NMAX, int LD, int ST, int TWM, int PAD, int PADIN,
          int R, int... Rest>
__device__ __forceinline__ void wave_passes(cpx<T>* x, int lane, const cpx<T>* tw, int n,
                                            WaveTab<T>& t) {
  if constexpr (sizeof...(Rest) == 0) {
    wave_pass<T, M, L, Ns, R, NMAX, LD, ST, TWM, PADIN, 0>(x, lane, tw, n, t);
  } else {
    constexpr int PO = Ns == 1 ? PAD : 0;
    wave_pass<T, M, L, Ns, R, NMAX, LD, ST_PLAIN, TWM, PADIN, PO>(x, lane, tw, n, t);
    wave_passes<T, M, L, Ns * R, NMAX, LD_PLAIN, ST, TWM, PAD, PO * R, Rest...>(x, lane, tw, n,
                                                                               t);
  }
}

template <int... Rs>
struct RadixProduct;
template <>
struct RadixProduct<> {
  static constexpr int value = 1;
};
template <int R, int... Rs>
struct RadixProduct<R, Rs...> {
  static constexpr int value = R * RadixProduct<Rs...>::value;
  static constexpr int first = R;
};

// A compile-time line plan: M-point FFTs with the given radices on L lanes
// per line; MODE 0: direct, n = M; MODE 1: Bluestein for any n <= NMAX =
// (M + 1) / 2; MODE 2: Rader, n = M + 1; PAD: keep the line padded between the
// first two passes.
template <int M, int L, int MODE, int TWM, int PAD, int... Rs>
struct WavePlan {
  static constexpr int n = 0, m = M, mode = MODE, lanes = L, twm = TWM;  // n: any
  static constexpr bool natural = false;
  // compiled for x and y lines too, up to 10 points a lane.  1024 points on 64 lanes (16
  // a lane) are slower than the engine's 128 threads: its fused x stage spills 291
  // registers in float32 and does not fit in float64 (gradre of 1024 x 1024 x 64: 6.93 /
  // 6.92 ms mixed / float64 on the engine, 9.14 / 11.67 here), and its 8 or 4 lines of
  // a y workgroup leave one workgroup on a CU (dual y pass of 1024 x 1024 x 100: 2.37 /
  // 4.97 against 2.96 / 6.19 ms).  In z it gains (128 x 128 x 1024, float64 step: 7.50 ->
  // 6.50 ms).
  static constexpr bool xy = MODE == 0 && M % 2 == 0 && (M + L - 1) / L <= 10;
  static constexpr int nmax = MODE == 1 ? (M + 1) / 2 : (MODE == 2 ? M + 1 : M);
  static constexpr int ldl = M + (PAD ? M / RadixProduct<Rs...>::first : 0) + 1;
  static_assert(RadixProduct<Rs...>::value == M, "radices do not multiply to M");
  static constexpr int tab = M + 5;  // LDS table: the passes' twiddles, then W_9^0..4
  static constexpr int npass = sizeof...(Rs);
  static constexpr int radix[npass] = {Rs...};
  // Lines per workgroup: the count that puts most lines on a CU (160 KB of
  // LDS, a twiddle table per workgroup), the larger one if another gains less
  // than a tenth (wider rows in the transposing kernels); 0: does not fit.
  static constexpr int lines(int csize) {
    const size_t extra = csize == 8 ? 4096 : 0;  // staged float64 boundary planes
    int best = 0, most = 0;
    for (int nl = 32; nl >= 4; nl >>= 1) {
      if (nl * L > 512 || nl * L < 64 || nl * csize < 64) continue;
      const size_t wg = (size_t(tab) + size_t(nl) * ldl) * csize + extra;
      if (wg > 160 * 1024) continue;
      const int on_cu = int(160 * 1024 / wg) * nl;
      if (on_cu * 10 > most * 11) {
        best = nl;
        most = on_cu;
      }
    }
    return best;
  }
  // waves per SIMD a kernel's registers should leave room for: what LDS allows, up to 4 in
  // float32 and 2 in float64
  static constexpr int waves(int csize) {
    const int nl = lines(csize) > 0 ? lines(csize) : 1;
    const size_t wg = (size_t(tab) + size_t(nl) * ldl) * csize;
    const int w = int(160 * 1024 / wg) * nl * L / 256;
    const int most = csize == 8 ? 4 : 2;
    return w < 1 ? 1 : (w > most ? most : w);
  }

  // Forward DFT of x[0..n) in place (x spans ldl elements).  Twiddles tw in
  // LDS; Bluestein filter and chirp (M entries each) and the Rader filter and
  // index tables perm (gather, then scatter) in global memory.
  template <typename T>
  static __device__ __forceinline__ void dft(cpx<T>* x, int lane, const cpx<T>* tw, int n,
                                             const cpx<T>* __restrict__ filt,
                                             const cpx<T>* __restrict__ chirp,
                                             const int* __restrict__ perm) {
    WaveTab<T> t;
    t.filt = filt;
    t.chirp = chirp;
    t.gin = perm;
    t.gout = perm + M;
    t.x0 = t.X0 = mkc<T>(0, 0);
    if constexpr (MODE == 0) {
      wave_passes<T, M, L, 1, M, LD_PLAIN, ST_PLAIN, TWM, PAD, 0, Rs...>(x, lane, tw, n, t);
    } else if constexpr (MODE == 1) {
      wave_passes<T, M, L, 1, nmax, LD_CHIRP, ST_FILTER, TWM, PAD, 0, Rs...>(x, lane, tw, n, t);
      wave_passes<T, M, L, 1, nmax, LD_PLAIN, ST_CHIRP, TWM, PAD, 0, Rs...>(x, lane, tw, n, t);
    } else {
      t.x0 = x[0];  // read by every lane before the first pass stores
      wave_passes<T, M, L, 1, M, LD_GATHER, ST_FILTER, TWM, PAD, 0, Rs...>(x, lane, tw, n, t);
      wave_passes<T, M, L, 1, M, LD_PLAIN, ST_SCATTER, TWM, PAD, 0, Rs...>(x, lane, tw, n, t);
      if (lane == 0) x[0] = t.X0;
    }
  }
};

// ---------------------------------------------------------------------------
// Plans of one DFT length on 64 lanes, twiddles in the order of W_M: the lines
// of the 512^3 and 1024^3 grids.  They keep their own passes because mixed runs
// on these grids keep their bits (see build_wave_fft): which of a complex
// product's two multiplies is fused depends on the code around it.
// ---------------------------------------------------------------------------
// Stage twiddles v[r] *= W_M^(r st), r = 1..R-1.  TWM 0: every factor read
// from the table; TWM 1: only W^st and W^(q st), q = ceil(sqrt(R)), are read
// and the others formed as W^(a + q b) = W^a W^(q b) (chains of at most
// about 2 sqrt(R) products: fewer LDS reads for some VALU work).
template <typename T, int R, int TWM>
__device__ __forceinline__ void fixed_twiddle(cpx<T>* v, const cpx<T>* tw, int st) {
  if constexpr (TWM == 0 || R <= 3) {
#pragma unroll
    for (int r = 1; r < R; ++r) v[r] = cmul(v[r], tw[r * st]);
  } else {
    constexpr int q = ceil_sqrt(R);
    cpx<T> w[R];
    w[1] = tw[st];
    if constexpr (q < R) w[q] = tw[q * st];
#pragma unroll
    for (int r = 2; r < R; ++r) {
      if (r == q) continue;
      const int a = r % q, b = r / q;
      if (b == 0) w[r] = cmul(w[r - 1], w[1]);
      else if (a == 0) w[r] = cmul(w[r - q], w[q]);
      else w[r] = cmul(w[b * q], w[a]);
    }
#pragma unroll
    for (int r = 1; r < R; ++r) v[r] = cmul(v[r], w[r]);
  }
}

// One in-place Stockham pass of radix R at stride Ns on the M-point line x
// (LDS), twiddle table tw (M entries).  LD / ST: the engine's load and store
// variants (chirp on load; filter or chirp on store).
template <typename T, int M, int Ns, int R, int LD, int ST, int TWM>
__device__ __forceinline__ void fixed_pass(cpx<T>* x, int lane, const cpx<T>* tw,
                                          const PassIO<T>& io, cpx<T>& X0) {
  constexpr int nb = M / R;
  constexpr int NR = (nb + 63) / 64;
  constexpr int tstep = M / (Ns * R);
  static_assert(M % R == 0, "radix does not divide the length");
  cpx<T> v[NR][R];
#pragma unroll
  for (int b = 0; b < NR; ++b) {
    const unsigned j = unsigned(lane) + 64u * b;
    if ((b + 1) * 64 <= nb || j < unsigned(nb)) {
      pass_load<T, R, LD>(v[b], x, int(j), nb, io);
      if constexpr (Ns > 1) fixed_twiddle<T, R, TWM>(v[b], tw, int(j % unsigned(Ns)) * tstep);
      WDft<T, R>::run(v[b]);
    }
  }
  wave_sync();
#pragma unroll
  for (int b = 0; b < NR; ++b) {
    const unsigned j = unsigned(lane) + 64u * b;
    if ((b + 1) * 64 <= nb || j < unsigned(nb)) {
      const int jm = Ns > 1 ? int(j % unsigned(Ns)) : 0;
      pass_store<T, R, ST>(x, v[b], (int(j) - jm) * R + jm, Ns, io, X0);
    }
  }
  wave_sync();
}

// The passes of one M-point FFT: the first loads with LD, the last stores
// with ST.
template <typename T, int M, int Ns, int LD, int ST, int TWM, int R, int... Rest>
__device__ __forceinline__ void fixed_passes(cpx<T>* x, int lane, const cpx<T>* tw,
                                            const PassIO<T>& io, cpx<T>& X0) {
  if constexpr (sizeof...(Rest) == 0) {
    fixed_pass<T, M, Ns, R, LD, ST, TWM>(x, lane, tw, io, X0);
  } else {
    fixed_pass<T, M, Ns, R, LD, ST_PLAIN, TWM>(x, lane, tw, io, X0);
    fixed_passes<T, M, Ns * R, LD_PLAIN, ST, TWM, Rest...>(x, lane, tw, io, X0);
  }
}

// A plan whose DFT length is fixed too: length N computed by M-point FFTs with the
// given radices (MODE 0: direct, M = N; MODE 1: Bluestein, M >= 2N-1), stage
// twiddles per TWM.
template <int N, int M, int MODE, int TWM, int... Rs>
struct FixedPlan {
  static constexpr int n = N, m = M, mode = MODE, lanes = 64, nmax = N, twm = TWM;
  static constexpr int ldl = M + 1, tab = M, npass = 0;
  static constexpr bool natural = true, xy = MODE == 0 && M % 2 == 0;
  static constexpr const int* radix = nullptr;
  static constexpr int lines(int csize) {
    return (size_t(M) + 8 * (size_t(M) + 1)) * csize <= 160 * 1024 ? 8 : 0;
  }
  static constexpr int waves(int csize) { return csize == 8 && lines(16) > 0 ? 4 : 1; }
  static_assert(RadixProduct<Rs...>::value == M, "radices do not multiply to M");
  static_assert(MODE == 0 ? M == N : M >= 2 * N - 1, "bad Bluestein length");

  // Forward DFT of x[0..N) in place (x spans M elements).  Twiddles tw in
  // LDS; Bluestein filter and chirp (the engine's tables) in global memory.
  template <typename T>
  static __device__ __forceinline__ void dft(cpx<T>* x, int lane, const cpx<T>* tw, int,
                                             const cpx<T>* __restrict__ filt,
                                             const cpx<T>* __restrict__ chirp,
                                             const int* __restrict__) {
    PassIO<T> io;
    io.n = N;
    io.gin = io.gout = nullptr;
    io.filt = filt;
    io.chirp = chirp;
    io.x0 = mkc<T>(0, 0);
    cpx<T> X0 = mkc<T>(0, 0);
    if constexpr (MODE == 0) {
      fixed_passes<T, M, 1, LD_PLAIN, ST_PLAIN, TWM, Rs...>(x, lane, tw, io, X0);
    } else {
      fixed_passes<T, M, 1, LD_CHIRP, ST_FILTER, TWM, Rs...>(x, lane, tw, io, X0);
      fixed_passes<T, M, 1, LD_PLAIN, ST_CHIRP, TWM, Rs...>(x, lane, tw, io, X0);
    }
  }
};

// The compiled wave plans.  A line plan (LineFFTHost) with wave = w >= 0 is
// launched with the kernel instances of radix-set code RS_WAVE + w.  CS: the
// element size a plan is compiled for (16 float64, 8 float32, 0 both).
//
// Radices and lanes from a sweep of in-place line DFTs (one read and one write
// of every line; ns per line, float64 / float32): lanes filled by M/R
// butterflies and first radices that are odd or padded count most -- Bluestein
// 512 as 8 8 8 padded 2.49 / 1.27 against 3.40 / 1.73 unpadded, 320 as 5 8 8 on
// 64 lanes 1.67 / 0.89 and as 20 16 on 32 lanes 1.73 / 0.84, 448 as 7 8 8 2.01 /
// 1.03, 640 as 20 8 4 3.71 / 1.80 against 10 8 8 3.98 / 2.15, 900 as 15 15 4
// 5.91 / 2.53 against 10 9 10 7.29 / 3.21.
// Plans of TWM 0 keep the radices and the order of the general engine: they
// give its bits, which mixed plans need (see build_wave_fft).
// Whole steps before and after the compiled lines, per-field launches merged in
// both: HD 32^3 float64 316 -> 262 us, 8 x HD 64^3 2.37 -> 2.14 ms, HD 192^3 mixed
// 3.59 -> 2.33 ms, HD 256^3 float64 14.5 -> 11.4 ms, Boussinesq 128^3 (d = 8) 4.0 ->
// 3.27 ms, rotating Boussinesq 96x144x150 mixed 1.57 -> 1.25 ms, MHD 128^3 3.41 ->
// 2.71 ms, gradre 256^3 mixed 1.91 -> 1.33 ms; the 160x120x103 transform 84.7 ->
// 76.8 us.
enum { RS_WAVE = 4 };
template <int W>
struct WavePlanN;
#define SPX_PLAN(W, CS, ...)                   \
  template <>                                  \
  struct WavePlanN<W> {                        \
    using type = __VA_ARGS__;                  \
    static constexpr int csize = CS;           \
  };
#define SPX_WAVE_PLAN(W, CS, ...) SPX_PLAN(W, CS, WavePlan<__VA_ARGS__>)
// nz = 512 + 25 (z lines of the 512^3 grids, d = 5): Bluestein on 1080 = 18 6 10
SPX_PLAN(0, 0, FixedPlan<537, 1080, 1, 1, 18, 6, 10>)
// nz = 512 + 27 (the 512^3 grids, d = 8): direct 539 = 11 7 7
SPX_PLAN(1, 0, FixedPlan<539, 539, 0, 1, 11, 7, 7>)
// nz = 1024 + 25 (the 1024^3 grids, d = 5): Bluestein on 2100 = 15 20 7, float32 only
SPX_PLAN(2, 8, FixedPlan<1049, 2100, 1, 1, 15, 20, 7>)
// 512-point x and y lines
SPX_PLAN(3, 0, FixedPlan<512, 512, 0, 1, 8, 8, 8>)
// direct lengths of x, y and (np + C) z lines, with the engine's radices
SPX_WAVE_PLAN(4, 0, 32, 4, 0, 0, 1, 4, 8)
SPX_WAVE_PLAN(5, 0, 48, 8, 0, 0, 1, 4, 4, 3)
SPX_WAVE_PLAN(6, 0, 64, 8, 0, 0, 1, 8, 8)
SPX_WAVE_PLAN(7, 0, 80, 16, 0, 0, 1, 4, 4, 5)
SPX_WAVE_PLAN(8, 0, 96, 16, 0, 0, 1, 4, 8, 3)
SPX_WAVE_PLAN(9, 0, 120, 16, 0, 0, 1, 8, 3, 5)
SPX_WAVE_PLAN(10, 0, 128, 16, 0, 0, 1, 4, 4, 8)
SPX_WAVE_PLAN(11, 0, 144, 16, 0, 0, 1, 4, 4, 9)
SPX_WAVE_PLAN(12, 0, 160, 32, 0, 0, 1, 4, 8, 5)
SPX_WAVE_PLAN(13, 0, 192, 32, 0, 0, 1, 8, 8, 3)
SPX_WAVE_PLAN(14, 0, 240, 32, 0, 0, 1, 4, 4, 3, 5)
SPX_WAVE_PLAN(15, 0, 256, 32, 0, 0, 1, 4, 8, 8)
SPX_WAVE_PLAN(16, 0, 288, 32, 0, 0, 1, 4, 8, 9)
SPX_WAVE_PLAN(17, 0, 320, 64, 0, 0, 1, 8, 8, 5)
SPX_WAVE_PLAN(18, 0, 384, 64, 0, 0, 1, 4, 4, 8, 3)
SPX_WAVE_PLAN(19, 0, 1024, 64, 0, 0, 1, 4, 4, 8, 8)
// Rader lengths with the engine's radices: 64 + 25 and 256 + 25 (d = 5)
SPX_WAVE_PLAN(20, 0, 88, 16, 2, 0, 1, 8, 11)
SPX_WAVE_PLAN(21, 0, 280, 64, 2, 0, 1, 8, 5, 7)
// Bluestein on the engine's own M and radices: z lines of 32 + 25, 128 + 25,
// 160 + 25, 192 + 25, 320 + 25, 384 + 25 and their neighbours
SPX_WAVE_PLAN(22, 0, 120, 16, 1, 0, 1, 8, 3, 5)
SPX_WAVE_PLAN(23, 0, 315, 64, 1, 0, 0, 9, 5, 7)
SPX_WAVE_PLAN(24, 0, 375, 64, 1, 0, 0, 3, 5, 5, 5)
SPX_WAVE_PLAN(25, 0, 441, 64, 1, 0, 0, 9, 7, 7)
SPX_WAVE_PLAN(26, 0, 700, 64, 1, 0, 1, 4, 5, 5, 7)
SPX_WAVE_PLAN(27, 0, 840, 64, 1, 0, 1, 8, 3, 5, 7)
// the ladder of Bluestein lengths for the z lines of float64 plans (no n <= 32
// needs one)
SPX_WAVE_PLAN(28, 16, 128, 16, 1, 2, 1, 16, 8)
SPX_WAVE_PLAN(29, 16, 192, 32, 1, 2, 1, 8, 4, 6)
SPX_WAVE_PLAN(30, 16, 256, 32, 1, 2, 1, 8, 8, 4)
SPX_WAVE_PLAN(31, 16, 320, 64, 1, 2, 0, 5, 8, 8)
SPX_WAVE_PLAN(32, 16, 384, 64, 1, 2, 0, 6, 8, 8)
SPX_WAVE_PLAN(33, 16, 448, 64, 1, 2, 0, 7, 8, 8)
SPX_WAVE_PLAN(34, 16, 512, 64, 1, 2, 1, 8, 8, 8)
SPX_WAVE_PLAN(35, 16, 640, 32, 1, 2, 1, 20, 8, 4)
SPX_WAVE_PLAN(36, 16, 720, 64, 1, 2, 0, 10, 6, 12)
SPX_WAVE_PLAN(37, 16, 900, 64, 1, 2, 0, 15, 15, 4)
SPX_WAVE_PLAN(38, 16, 1080, 64, 1, 2, 0, 18, 6, 10)
// odd direct lengths, z lines only: np + 25 of 80, 96, 100, 144, 150 and 200 planes,
// np + 27 of 48 and 64, with the engine's radices (z stages of an RK stage on the
// engine and compiled: 16 members of 64^2 x 91 float64 201 + 148 -> 147 + 85 us,
// 96x144x175 mixed 68 + 46 -> 40 + 31 us)
SPX_WAVE_PLAN(39, 0, 75, 16, 0, 0, 0, 3, 5, 5)
SPX_WAVE_PLAN(40, 0, 91, 16, 0, 0, 0, 7, 13)
SPX_WAVE_PLAN(41, 0, 105, 16, 0, 0, 0, 3, 5, 7)
SPX_WAVE_PLAN(42, 0, 121, 16, 0, 0, 0, 11, 11)
SPX_WAVE_PLAN(43, 0, 125, 32, 0, 0, 0, 5, 5, 5)
SPX_WAVE_PLAN(44, 0, 169, 16, 0, 0, 0, 13, 13)
SPX_WAVE_PLAN(45, 0, 175, 32, 0, 0, 0, 5, 5, 7)
SPX_WAVE_PLAN(46, 0, 225, 32, 0, 0, 0, 9, 5, 5)
// further even direct lengths, with the engine's radices (transforms of
// 180x24x88 both ways on the engine 45.2 us, here 32.8; HD step of 108x34x49
// float64 253 -> 233 us)
SPX_WAVE_PLAN(47, 0, 24, 4, 0, 0, 1, 8, 3)
SPX_WAVE_PLAN(48, 0, 40, 8, 0, 0, 1, 8, 5)
SPX_WAVE_PLAN(49, 0, 60, 16, 0, 0, 1, 4, 3, 5)
SPX_WAVE_PLAN(50, 0, 72, 8, 0, 0, 1, 8, 9)
SPX_WAVE_PLAN(51, 0, 88, 16, 0, 0, 1, 8, 11)
SPX_WAVE_PLAN(52, 0, 90, 16, 0, 0, 0, 2, 9, 5)
SPX_WAVE_PLAN(53, 0, 100, 32, 0, 0, 1, 4, 5, 5)
SPX_WAVE_PLAN(54, 0, 108, 16, 0, 0, 1, 4, 9, 3)
SPX_WAVE_PLAN(55, 0, 180, 32, 0, 0, 1, 4, 9, 5)
SPX_WAVE_PLAN(56, 0, 200, 32, 0, 0, 1, 8, 5, 5)
#undef SPX_WAVE_PLAN
#undef SPX_PLAN
constexpr int kWavePlans = 57;
template <int RS>
struct WavePlanOf {
  using type = typename WavePlanN<RS - RS_WAVE>::type;
};
// lines per workgroup of plan W for csize-byte elements, 0: not compiled for them
template <int W>
constexpr int wave_lines(int csize) {
  using N = WavePlanN<W>;
  return N::csize && N::csize != csize ? 0 : N::type::lines(csize);
}

}  // namespace spx

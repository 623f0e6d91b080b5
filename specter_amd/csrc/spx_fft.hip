// Line-FFT kernels of libspx: x (real<->half-complex), y, z (with the FC
// continuation and the (kx,y,z)<->(z,y,kx) transposes fused in), the fused
// gradient-product x pass of gradre/advect, and the z-line kernels of the
// boundary / projection / diagnostics stages.
//
// Build: the host part of this file is compiled in parts so that the kernel
// instantiations build in parallel (SPX_PART = 1: plan tables, in-place z
// transforms and the entry points of the passes, 3: boundary and projection
// launchers, 16: magnetic walls and pressure, 8: diagnostics; in float64 / float32 4 / 5: forward z pass, 6 / 7:
// backward z pass, 2 / 9: y pass, 10 / 11: x passes, 12 / 13 and 14 / 15:
// gradient products); without SPX_PART everything is compiled in one unit.
//
// Precision: the transform kernels are templated on their arithmetic / buffer
// type T (double; float for the nonlinear pipeline of mixed-precision plans,
// where the first z pass reads the float64 state, TI = double).  The
// boundary, projection and diagnostics kernels compute in float64; they are
// templated on the storage type TS of the fields and instantiated for double.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <cstdint>
#include <thread>
#include <unordered_map>

#include "spx_engine.h"
#include "spx_wave.h"

namespace spx {

// (0,1)*k*v evaluated as the reference's complex product (-k Im v, k Re v)
template <typename T>
__device__ __forceinline__ cpx<T> ikmul(T k, cpx<T> v) { return mkc<T>(-(k * v.y), k * v.x); }

template <typename TO, typename TI>
__device__ __forceinline__ cpx<TO> ccast(cpx<TI> v) { return mkc<TO>(TO(v.x), TO(v.y)); }

// Twiddles at the head of dynamic LDS, then the line buffers.  Each thread
// belongs to line `line` (lane `lane` of tpl); xl is its line buffer.
#define SPX_PROLOGUE(CT, f)                                      \
  extern __shared__ unsigned char smem[];                        \
  CT* const tws = reinterpret_cast<CT*>(smem);                   \
  CT* const lds = tws + (f).tab;                                 \
  stage_twiddles<RS>(tws, (f));                                   \
  const int tid = threadIdx.x;                                   \
  const int line = tid >> (f).lgtpl, lane = tid & ((f).tpl - 1); \
  CT* const xl = lds + line * (f).ldl;                           \
  (void)xl;

constexpr int KEEP = kStage;  // line elements a thread can hold in registers (n <= KEEP*tpl)
// Workgroups hold nl lines of tpl threads: 256 threads, or one line of up to
// 512 threads for the longest lines (e.g. Bluestein length 2100 for nz = 1049).
constexpr int kMaxBlock = 512;

// Forward DFT of a z line in LDS: the compiled wave plan for radix-set codes
// RS_WAVE + w (tables: twiddles staged in LDS, filter and chirp global),
// the general engine otherwise.  Ends with a workgroup barrier either way.
template <typename T, int RS>
__device__ __forceinline__ void zline_dft(cpx<T>* x, const LineFFT<cpx<T>>& f, const cpx<T>* tw,
                                          int lane) {
  if constexpr (RS >= RS_WAVE) {
    using P = typename WavePlanOf<RS>::type;
    P::template dft<T>(x, lane, tw, f.n, f.bfil, f.chirp, f.perm);
    __syncthreads();
  } else {
    line_dft<T, RS>(x, f, tw, lane);
  }
}

// Forward FFT of a direct (mode 0) line without the closing workgroup
// barrier: the caller synchronises the line (line_sync); the wave plan or
// the engine's passes.
template <typename T, int RS>
__device__ __forceinline__ void line_fft_nosync(cpx<T>* x, const LineFFT<cpx<T>>& f,
                                                const cpx<T>* tw, int lane) {
  if constexpr (RS >= RS_WAVE) {
    using P = typename WavePlanOf<RS>::type;
    static_assert(P::mode == 0, "direct plans only");
    P::template dft<T>(x, lane, tw, f.n, nullptr, nullptr, nullptr);
  } else {
    fft_lds<T, RS>(x, f, tw, lane);
  }
}

// line elements a thread holds in registers in the z kernels (n <= KN * tpl)
template <int RS>
constexpr int keep_n() {
  if constexpr (RS >= RS_WAVE) {
    using P = typename WavePlanOf<RS>::type;
    return (P::nmax + P::lanes - 1) / P::lanes;
  } else {
    return KEEP;
  }
}

// waves per SIMD of a line kernel's register budget (compiled plans: what
// their LDS leaves room for)
template <typename T, int RS>
constexpr int min_waves() {
  if constexpr (RS >= RS_WAVE) return WavePlanOf<RS>::type::waves(2 * sizeof(T));
  else return 1;
}

// idx = first, first + step, ... < count: wr(idx, rd(idx)).  KN > 0 (the
// compiled plans, count <= first + KN*step): every LDS read is issued before
// the first global store instead of one read-wait-store round trip each.
template <int KN, typename V, typename Rd, typename Wr>
__device__ __forceinline__ void lds_to_global(int first, int step, int count, Rd rd, Wr wr) {
  if constexpr (KN > 0) {
    V v[KN];
#pragma unroll
    for (int q = 0; q < KN; ++q) {
      const int idx = first + q * step;
      if (idx < count) v[q] = rd(idx);
    }
#pragma unroll
    for (int q = 0; q < KN; ++q) {
      const int idx = first + q * step;
      if (idx < count) wr(idx, v[q]);
    }
  } else {
    for (int idx = first; idx < count; idx += step) wr(idx, rd(idx));
  }
}

// XCD-aware order of the tiles along gridDim.x.  Workgroups are handed to the
// 8 XCDs (each with its own L2) round-robin by linear id; the tiles of the
// transposing kernels are about as wide as a cache line and not aligned to
// one, so neighbouring tiles must meet in one L2.  Each XCD gets a contiguous
// range of logical tiles (a bijection on [0, gridDim.x)).
__device__ __forceinline__ unsigned xcd_tile() {
  constexpr unsigned X = 8;
  const unsigned n = gridDim.x, pid = blockIdx.x;
  const unsigned q = n / X, r = n % X;
  const unsigned x = pid % X, slot = pid / X;
  return x * q + (x < r ? x : r) + slot;
}

// Up to kMaxComp fields of one launch (blockIdx.y selects): the components
// of a vector field go through one launch, so a small grid fills the GPU and
// a stage has a third of the launches.  With the products' half spectra taken
// in the x stage (24 launches per HD stage before, 9 now) an RK2 step of 32^3
// takes 318 us instead of 529, Boussinesq 128^3 RK4 4.01 ms instead of 4.98,
// MHD 128^3 RK2 3.42 ms instead of 4.21, HD 256^3 RK4 14.6 ms instead of 15.4.
// The kernels read their field's pointers ahead of the prologue, together with its
// own arguments: after it, their cold reads were two to four percent of a small
// launch (transforms both ways on the engine's lines, us: 36x30x65 38.4 -> 36.9,
// 54x56x71 47.8 -> 46.2, 28x26x49 41.7 -> 39.6, 110x98x110 79.3 -> 77.1).
constexpr int kMaxComp = 8;

// ---------------------------------------------------------------------------
// z transforms in place on S (contiguous lines)
// ---------------------------------------------------------------------------
template <typename T, int RS>
__global__ void __launch_bounds__(kMaxBlock) k_z_inplace(cpx<T>* __restrict__ S, long nlines,
                                                   LineFFT<cpx<T>> f, int np, int forward,
                                                   int cont, double scale,
                                                   const double* __restrict__ dir, int C,
                                                   int d) {
  using Cp = cpx<T>;
  SPX_PROLOGUE(Cp, f);
  const int n = f.n;
  const long ln = long(blockIdx.x) * f.nl + line;
  const bool ok = ln < nlines;
  const int nload = (forward && cont) ? np : n;
  for (int k = lane; k < nload; k += f.tpl) {
    Cp v = ok ? S[ln * n + k] : mkc<T>(0, 0);
    if (!forward) v.y = -v.y;
    xl[k] = v;
  }
  __syncthreads();
  if (forward && cont) {
    fc_continue_lds(lds, f.nl, f.ldl, np, C, d, dir);
    __syncthreads();
  }
  zline_dft<T, RS>(xl, f, tws, lane);
  if (ok) {
    for (int k = lane; k < n; k += f.tpl) {
      Cp v = xl[k];
      if (!forward) {
        v.y = -v.y;
        if (k < np && scale != 1.0) v = cscale(v, T(scale));
      }
      S[ln * n + k] = v;
    }
  }
}

// Continuation only (fftp.fpp:755-773), in place on S, float64 arithmetic.
template <typename T>
__global__ void k_fc_continue(cpx<T>* __restrict__ S, long nlines, int n, int np, int C, int d,
                              const double* __restrict__ dir) {
#pragma clang fp contract(off)
  const long e = long(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= nlines * C) return;
  const long ln = e / C;
  const int ii = int(e - ln * C);
  const cpx<T>* x = S + ln * n;
  const int top = np - d;
  const double* D0 = dir + ii * d;
  const double* D1 = dir + (C - 1 - ii) * d;
  double ar = D0[0] * double(x[top].x) + D1[0] * double(x[d - 1].x);
  double ai = D0[0] * double(x[top].y) + D1[0] * double(x[d - 1].y);
  for (int jj = 1; jj < d; ++jj) {
    ar = ar + D0[jj] * double(x[top + jj].x);
    ar = ar + D1[jj] * double(x[d - 1 - jj].x);
    ai = ai + D0[jj] * double(x[top + jj].y);
    ai = ai + D1[jj] * double(x[d - 1 - jj].y);
  }
  S[ln * n + np + ii] = mkc<T>(T(ar), T(ai));
}

// ---------------------------------------------------------------------------
// forward 3D last pass: X(kx,y,z) planes < np -> continuation -> z FFT -> S(z,y,kx)
// blockIdx.z = member: S advances by n*ny*nkx, X by xstride elements per member.
// The lines of a workgroup are nl consecutive (kx, y) points e = kx + nkx*y of
// a plane, whatever nkx is: tiles over kx alone left 15 of 32 lines of a
// 17-point row (nx = 32) empty, 3 of 36 of a 33-point one.
// ---------------------------------------------------------------------------
template <typename T>
struct ZX2S {
  const cpx<T>* x[kMaxComp];
  cpx<T>* s[kMaxComp];
  const cpx<double>* xb[kMaxComp];
};

// BND (mixed plans): the 2d boundary planes z = 0..d-1, np-d..np-1 come in
// float64 from xb (planes [member][q][ky][kx], q < 2d) and the continuation
// is evaluated from them, so the float32 roundoff of the other planes is not
// amplified by the continuation.
template <typename T, int RS, bool BND>
__global__ void __launch_bounds__(kMaxBlock, (min_waves<T, RS>())) k_z_x2s(ZX2S<T> a, LineFFT<cpx<T>> f, int nkx,
                                               int ny, int np, int nofft,
                                               const double* __restrict__ dir, int C, int d,
                                               long xstride) {
  using Cp = cpx<T>;
  const Cp* __restrict__ X = a.x[blockIdx.y] + blockIdx.z * xstride;
  Cp* __restrict__ S = a.s[blockIdx.y];
  SPX_PROLOGUE(Cp, f);
  const int n = f.n;
  const long pl = long(nkx) * ny;
  S += blockIdx.z * (pl * n);
  const int e0 = int(xcd_tile()) * f.nl;
  const int nlines = int(pl);
  const int nload = nofft ? n : np;
  {
    const int l = tid & (f.nl - 1), e = e0 + l;
    if constexpr (RS >= RS_WAVE) {
      // compiled plans (n <= KN*tpl): the thread's loads in flight together
      constexpr int KN = keep_n<RS>();
      Cp v[KN];
#pragma unroll
      for (int q = 0; q < KN; ++q) {
        const int k = (tid >> f.lgnl) + q * f.tpl;
        v[q] = mkc<T>(0, 0);
        if (e < nlines && k < nload) v[q] = X[e + pl * k];
      }
#pragma unroll
      for (int q = 0; q < KN; ++q) {
        const int k = (tid >> f.lgnl) + q * f.tpl;
        if (k < nload) lds[l * f.ldl + k] = v[q];
      }
    } else {
      for (int k = tid >> f.lgnl; k < nload; k += f.tpl) {
        Cp v = mkc<T>(0, 0);
        if (e < nlines) v = X[e + pl * k];
        lds[l * f.ldl + k] = v;
      }
    }
  }
  __syncthreads();
  if (!nofft) {
    if constexpr (BND) {
#pragma clang fp contract(off)
      const int d2 = 2 * d;
      const cpx<double>* xb = a.xb[blockIdx.y] + blockIdx.z * (pl * d2);
      // the tile's float64 boundary values, staged once behind the line
      // buffers (16-byte aligned; bnd_stage_bytes at launch): bl[l * d2 + q]
      cpx<double>* const bl = reinterpret_cast<cpx<double>*>(
          (reinterpret_cast<uintptr_t>(lds + f.nl * f.ldl) + 15) & ~uintptr_t(15));
      for (int t = tid; t < f.nl * d2; t += blockDim.x) {
        const int q = t >> f.lgnl, l = t & (f.nl - 1), e = e0 + l;
        const int z = q < d ? q : np - d2 + q;
        const cpx<double> v = e < nlines ? xb[e + pl * q] : mkc<double>(0, 0);
        // (a point of both blocks, np < 2d, is the top one's)
        if (q >= d || z < np - d) lds[l * f.ldl + z] = mkc<T>(T(v.x), T(v.y));
        bl[l * d2 + q] = v;
      }
      __syncthreads();
      // continuation (fftp.fpp:755-773 order): x[top+jj] is plane q = d+jj,
      // x[d-1-jj] is plane q = d-1-jj
      for (int t = tid; t < f.nl * C; t += blockDim.x) {
        const int l = t / C, ii = t - l * C;
        const cpx<double>* bq = bl + l * d2;
        const double* D0 = dir + ii * d;
        const double* D1 = dir + (C - 1 - ii) * d;
        const cpx<double> t0 = bq[d], b0 = bq[d - 1];
        double ar = D0[0] * t0.x + D1[0] * b0.x;
        double ai = D0[0] * t0.y + D1[0] * b0.y;
        for (int jj = 1; jj < d; ++jj) {
          const cpx<double> ut = bq[d + jj], ub = bq[d - 1 - jj];
          ar = ar + D0[jj] * ut.x;
          ar = ar + D1[jj] * ub.x;
          ai = ai + D0[jj] * ut.y;
          ai = ai + D1[jj] * ub.y;
        }
        lds[l * f.ldl + np + ii] = mkc<T>(T(ar), T(ai));
      }
      __syncthreads();
    } else if (C > 0) {
      fc_continue_lds(lds, f.nl, f.ldl, np, C, d, dir);
      __syncthreads();
    }
    zline_dft<T, RS>(xl, f, tws, lane);
  }
  const int e = e0 + line;
  if (e < nlines) {
    const int j = e / nkx, i = e - j * nkx;
    Cp* so = S + long(n) * (j + long(ny) * i);
    lds_to_global<0, Cp>(lane, f.tpl, n, [&](int k) { return xl[k]; },
                         [&](int k, Cp v) { so[k] = v; });
  }
}

// ---------------------------------------------------------------------------
// float64 values of the backward z transform at the 2d boundary planes
// z = 0..d-1 and np-d..np-1 (the points the FC continuation reads), for the
// float32 nonlinear pipeline of mixed plans: a direct partial DFT of every
// line, 16 lanes per line (4 lines per wavefront), for v and (i kz) v
// together.  Twiddles: w1[k] = exp(+2 pi i k/n) and wt[k] = exp(+2 pi i k
// (np-d)/n) from long-double tables, then exp(+2 pi i k z/n) for the d
// consecutive z of each wall block by d-1 products (error ~ d ulp).
// blockIdx.y = component.  Output planes [comp][member][q][ky][kx].
// ---------------------------------------------------------------------------
struct BndSrc {
  const cpx<double>* s[4];
};

template <int D, int U>
__global__ void __launch_bounds__(256) k_z_s2x_bnd(BndSrc src, cpx<double>* __restrict__ XVb,
                                                   cpx<double>* __restrict__ XZb,
                                                   const cpx<double>* __restrict__ w1,
                                                   const cpx<double>* __restrict__ wt, int n,
                                                   int nkx, int ny, int mem,
                                                   const double* __restrict__ kz) {
  constexpr int D2 = 2 * D;
  constexpr int LPL = 16;  // lanes per line
  const int sub = threadIdx.x & (LPL - 1);
  const long nlines = long(nkx) * ny;
  const long ln = long(blockIdx.x) * (blockDim.x / LPL) + (threadIdx.x / LPL);
  const bool ok = ln < nlines * mem;
  const int comp = blockIdx.y;
  const cpx<double>* S = src.s[comp] + (ok ? ln : 0) * n;
  const long b = ok ? ln / nlines : 0, l = ok ? ln - b * nlines : 0;
  const long i = l / ny, jy = l - i * ny;
  const long o = ((long(comp) * mem + b) * D2) * nlines + jy * nkx + i;
  // v and (i kz) v from one load of the line.  The top block uses
  // exp(+2 pi i k (np-d+q)/n) = wt[k] exp(+2 pi i k q/n): both blocks share
  // the twiddle recurrence, the top one on u_k = v_k wt[k].
  cpx<double> acc[2][D2];
#pragma unroll
  for (int kind = 0; kind < 2; ++kind)
#pragma unroll
    for (int q = 0; q < D2; ++q) acc[kind][q] = mkc<double>(0, 0);
  if (ok) {
    // U points per lane in flight: their loads first (indices past the line
    // end clamped to 0 and their values zeroed), then the sums in the same
    // point order as one point at a time (HD 512^3, d = 5: U = 2 1.17 ms per
    // launch, U = 1 1.25, U = 4 1.27 at two waves per SIMD)
    for (int k0 = sub; k0 < n; k0 += U * LPL) {
      cpx<double> vv[U], ww[U], ss[U];
      double kk[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u * LPL;
        const int kc = k < n ? k : 0;
        vv[u] = S[kc];
        kk[u] = kz[kc];
        ww[u] = wt[kc];
        ss[u] = w1[kc];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool in = k0 + u * LPL < n;
        const cpx<double> v0 = in ? vv[u] : mkc<double>(0, 0);
        const cpx<double> v1 = ikmul(kk[u], v0);
        const cpx<double> wtk = ww[u];
        const cpx<double> u0 = cmul(v0, wtk), u1 = cmul(v1, wtk);
        const cpx<double> step = ss[u];
        cpx<double> t = mkc<double>(1.0, 0.0);
#pragma unroll
        for (int q = 0; q < D; ++q) {
          acc[0][q] = cadd(acc[0][q], cmul(v0, t));
          acc[0][D + q] = cadd(acc[0][D + q], cmul(u0, t));
          acc[1][q] = cadd(acc[1][q], cmul(v1, t));
          acc[1][D + q] = cadd(acc[1][D + q], cmul(u1, t));
          if (q + 1 < D) t = cmul(t, step);
        }
      }
    }
  }
  // reduce over the 16 lanes of the line (lanes of one line are contiguous)
#pragma unroll
  for (int kind = 0; kind < 2; ++kind) {
#pragma unroll
    for (int off = LPL / 2; off > 0; off >>= 1) {
#pragma unroll
      for (int q = 0; q < D2; ++q) {
        acc[kind][q].x += __shfl_xor(acc[kind][q].x, off);
        acc[kind][q].y += __shfl_xor(acc[kind][q].y, off);
      }
    }
    if (ok) {
      cpx<double>* out = kind ? XZb : XVb;
#pragma unroll
      for (int q = 0; q < D2; ++q)
        if (sub == q) out[o + q * nlines] = acc[kind][q];
    }
  }
}

// ---------------------------------------------------------------------------
// backward 3D first pass: S * (i k_dir) -> z IFFT -> X planes < nzout.
// DUAL: the same load also gives X2 <- z IFFT of (i kz) S.
// blockIdx.z = member: S advances by n*ny*nkx, X and X2 by nkx*ny*nzout.
// Lines as in k_z_x2s.
// ---------------------------------------------------------------------------
template <typename T, typename TI>
struct ZS2X {
  const cpx<TI>* s[kMaxComp];
  cpx<T>* x[kMaxComp];
  cpx<T>* x2[kMaxComp];
};

template <typename T, int RS, bool DUAL, typename TI>
__global__ void __launch_bounds__(kMaxBlock, (min_waves<T, RS>())) k_z_s2x(ZS2X<T, TI> a, LineFFT<cpx<T>> f, int nkx,
                                               int ny, int nzout, int dirn, int nofft,
                                               const double* __restrict__ kx,
                                               const double* __restrict__ ky,
                                               const double* __restrict__ kz) {
  using Cp = cpx<T>;
  const cpx<TI>* __restrict__ S = a.s[blockIdx.y];
  Cp* __restrict__ X = a.x[blockIdx.y];
  SPX_PROLOGUE(Cp, f);
  const int n = f.n;
  const long pl = long(nkx) * ny;
  S += blockIdx.z * (pl * n);
  const int e0 = int(xcd_tile()) * f.nl;
  const int nlines = int(pl);
  const bool ok = e0 + line < nlines;
  const int j = ok ? (e0 + line) / nkx : 0, i = ok ? e0 + line - j * nkx : 0;
  const long base = long(n) * (j + long(ny) * i);
  // the line (times i k_dirn).  The dual transform needs it again: float
  // kernels and the wave plans (whose occupancy LDS bounds) keep it in
  // registers, the other float64 kernels read it again (the second read hits
  // in L2 and keeps the registers free for occupancy)
  constexpr bool KEEPV = DUAL && (sizeof(T) == 4 || RS >= RS_WAVE);
  constexpr int KN = keep_n<RS>();
  auto load = [&](int k) {
    Cp v = mkc<T>(0, 0);
    if (ok) {
      v = ccast<T>(S[base + k]);
      if (dirn == 1) v = ikmul(T(kx[i]), v);
      else if (dirn == 2) v = ikmul(T(ky[j]), v);
      else if (dirn == 3) v = ikmul(T(kz[k]), v);
    }
    return v;
  };
  Cp keep[KEEPV ? KN : 1];
  if constexpr (RS >= RS_WAVE) {
    // compiled plans: the line's raw values (and kz) in flight together, then
    // the derivative factor and the LDS writes
    cpx<TI> raw[KN];
    double kzv[KN];
    const double kline = (ok && dirn == 1) ? kx[i] : ((ok && dirn == 2) ? ky[j] : 0.0);
#pragma unroll
    for (int q = 0; q < KN; ++q) {
      const int k = lane + q * f.tpl;
      raw[q] = mkc<TI>(0, 0);
      kzv[q] = kline;
      if (ok && k < n) {
        raw[q] = S[base + k];
        if (dirn == 3) kzv[q] = kz[k];
      }
    }
#pragma unroll
    for (int q = 0; q < KN; ++q) {
      const int k = lane + q * f.tpl;
      if (k < n) {
        Cp v = ccast<T>(raw[q]);
        if (ok && dirn != 0) v = ikmul(T(kzv[q]), v);
        if constexpr (KEEPV) keep[q] = v;
        xl[k] = cconj(v);
      }
    }
  } else {
#pragma unroll
    for (int q = 0; q < KN; ++q) {
      const int k = lane + q * f.tpl;
      if (k < n) {
        const Cp v = load(k);
        if constexpr (KEEPV) keep[q] = v;
        xl[k] = cconj(v);
      }
    }
  }
  __syncthreads();
  if (!nofft) zline_dft<T, RS>(xl, f, tws, lane);
  const int l = tid & (f.nl - 1), e = e0 + l;
  // (batched stores measured slower here: the z line kernels are VALU-bound)
  constexpr int KB = 0;
  if (e < nlines) {
    Cp* __restrict__ xo = X + blockIdx.z * (pl * nzout) + e;
    lds_to_global<KB, Cp>(
        tid >> f.lgnl, f.tpl, nzout, [&](int k) { return cconj(lds[l * f.ldl + k]); },
        [&](int k, Cp v) { xo[pl * k] = v; });
  }
  if constexpr (DUAL) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < KN; ++q) {
      const int k = lane + q * f.tpl;
      if (k < n) {
        if constexpr (KEEPV) xl[k] = cconj(ikmul(T(kz[k]), keep[q]));
        else xl[k] = cconj(ikmul(T(kz[k]), load(k)));
      }
    }
    __syncthreads();
    zline_dft<T, RS>(xl, f, tws, lane);
    if (e < nlines) {
      Cp* __restrict__ xo = a.x2[blockIdx.y] + blockIdx.z * (pl * nzout) + e;
      lds_to_global<KB, Cp>(
          tid >> f.lgnl, f.tpl, nzout, [&](int k) { return cconj(lds[l * f.ldl + k]); },
          [&](int k, Cp v) { xo[pl * k] = v; });
    }
  }
}

// ---------------------------------------------------------------------------
// y transform of X (lines along y, stride nkx).  The lines of all planes are
// counted through, e = kx + nkx*plane, and a workgroup takes nl consecutive
// ones, so only the last workgroup of a field has empty lines.  blockIdx.y:
// field.  y2 of a field (DUAL kernels, backward): also y2 <- y IFFT of
// (i ky) in from the same load; null: not for this field.
// Cy > 0 (forward): FC-Gram continuation of each line before the FFT
// (fftp.fpp:565-581): rows npy..ny-1 from rows 0..oy-1 and npy-oy..npy-1.
// ---------------------------------------------------------------------------
template <typename T>
struct YFields {
  const cpx<T>* in[kMaxComp];
  cpx<T>* out[kMaxComp];
  cpx<T>* y2[kMaxComp];
};

template <typename T, int RS, bool DUAL>
__global__ void __launch_bounds__(kMaxBlock, (min_waves<T, RS>())) k_y(YFields<T> a, LineFFT<cpx<T>> f, int nkx,
                                           int ny, long nlines, int forward,
                                           const double* __restrict__ ky, int npy, int Cy, int oy,
                                           const double* __restrict__ diry) {
  using Cp = cpx<T>;
  const Cp* const Xin = a.in[blockIdx.y];
  Cp* const Xout = a.out[blockIdx.y];
  SPX_PROLOGUE(Cp, f);
  const int l = tid & (f.nl - 1);
  const long e = long(xcd_tile()) * f.nl + l;
  const bool in = e < nlines;
  // (a 64-bit division only where the count needs it)
  const long plane = !in ? 0 : (nlines >> 32 ? e / nkx : long(unsigned(e) / unsigned(nkx)));
  const long base = plane * nkx * ny + (in ? e - plane * nkx : 0);
  const bool cont = forward && Cy > 0;
  const int nload = cont ? npy : ny;
  if constexpr (RS >= RS_WAVE) {
    // compiled plans (ny <= KN*tpl): all of a thread's loads in
    // flight at once instead of one load-wait-store round trip per element
    constexpr int KN = keep_n<RS>();
    Cp v[KN];
#pragma unroll
    for (int q = 0; q < KN; ++q) {
      const int jy = (tid >> f.lgnl) + q * f.tpl;
      v[q] = mkc<T>(0, 0);
      if (in && jy < nload) v[q] = Xin[base + long(nkx) * jy];
    }
#pragma unroll
    for (int q = 0; q < KN; ++q) {
      const int jy = (tid >> f.lgnl) + q * f.tpl;
      if (!forward) v[q].y = -v[q].y;
      if (jy < nload) lds[l * f.ldl + jy] = v[q];
    }
  } else {
    for (int jy = tid >> f.lgnl; jy < nload; jy += f.tpl) {
      Cp v = mkc<T>(0, 0);
      if (in) v = Xin[base + long(nkx) * jy];
      if (!forward) v.y = -v.y;
      lds[l * f.ldl + jy] = v;
    }
  }
  __syncthreads();
  if (cont) {
    fc_continue_lds(lds, f.nl, f.ldl, npy, Cy, oy, diry);
    __syncthreads();
  }
  constexpr int KN = keep_n<RS>();
  Cp keep[DUAL ? KN : 1];
  if constexpr (DUAL) {
#pragma unroll
    for (int q = 0; q < KN; ++q) {
      const int k = lane + q * f.tpl;
      if (k < ny) keep[q] = xl[k];
    }
  }
  zline_dft<T, RS>(xl, f, tws, lane);
  constexpr int KB = RS >= RS_WAVE ? keep_n<RS>() : 0;
  if (in) {
    Cp* xo = Xout + base;
    lds_to_global<KB, Cp>(
        tid >> f.lgnl, f.tpl, ny,
        [&](int jy) {
          Cp v = lds[l * f.ldl + jy];
          if (!forward) v.y = -v.y;
          return v;
        },
        [&](int jy, Cp v) { xo[long(nkx) * jy] = v; });
  }
  if constexpr (DUAL) {
    if (!a.y2[blockIdx.y]) return;  // uniform per workgroup
    __syncthreads();
#pragma unroll
    for (int q = 0; q < KN; ++q) {
      const int k = lane + q * f.tpl;
      if (k < ny) xl[k] = cconj(ikmul(T(ky[k]), cconj(keep[q])));
    }
    __syncthreads();
    zline_dft<T, RS>(xl, f, tws, lane);
    if (in) {
      Cp* yo = a.y2[blockIdx.y] + base;
      lds_to_global<KB, Cp>(
          tid >> f.lgnl, f.tpl, ny, [&](int jy) { return cconj(lds[l * f.ldl + jy]); },
          [&](int jy, Cp v) { yo[long(nkx) * jy] = v; });
    }
  }
}

// The half spectra of a row pair from the transform xl of A + iB.
template <typename T>
__device__ __forceinline__ void store_r2c_pair(const cpx<T>* xl, cpx<T>* o0, int nkx, int nx,
                                               int lane, int tpl) {
  const T h = T(0.5);
  for (int k = lane; k < nkx; k += tpl) {
    const cpx<T> Z = xl[k];
    const cpx<T> Zc = xl[k == 0 ? 0 : nx - k];
    o0[k] = mkc<T>((Z.x + Zc.x) * h, (Z.y - Zc.y) * h);
    o0[k + nkx] = mkc<T>((Z.y + Zc.y) * h, -(Z.x - Zc.x) * h);
  }
}

// ---------------------------------------------------------------------------
// x real -> half complex: rows 2p, 2p+1 packed as one complex line
// ---------------------------------------------------------------------------
// (blockIdx.y: field)
template <typename T>
struct XFields {
  const void* in[kMaxComp];
  void* out[kMaxComp];
};

template <int RS>
__global__ void __launch_bounds__(kMaxBlock) k_xr2c(XFields<double> a, LineFFT<cpx<double>> f,
                                              int nkx, long npairs) {
  using T = double;
  using Cp = cpx<T>;
  const T* __restrict__ R = static_cast<const T*>(a.in[blockIdx.y]);
  Cp* __restrict__ X = static_cast<Cp*>(a.out[blockIdx.y]);
  SPX_PROLOGUE(Cp, f);
  const int nx = f.n;
  const long p = long(blockIdx.x) * f.nl + line;
  const bool ok = p < npairs;
  const T* r0 = R + long(nx) * (2 * (ok ? p : 0));
  if constexpr (RS >= RS_WAVE) {  // batched loads
    constexpr int KN = keep_n<RS>();
    T a[KN], b[KN];
#pragma unroll
    for (int q = 0; q < KN; ++q) {
      const int x = lane + q * f.tpl;
      a[q] = b[q] = T(0);
      if (ok && x < nx) {
        a[q] = r0[x];
        b[q] = r0[x + nx];
      }
    }
#pragma unroll
    for (int q = 0; q < KN; ++q) {
      const int x = lane + q * f.tpl;
      if (x < nx) xl[x] = mkc<T>(a[q], b[q]);
    }
  } else {
    for (int x = lane; x < nx; x += f.tpl) xl[x] = ok ? mkc<T>(r0[x], r0[x + nx]) : mkc<T>(0, 0);
  }
  __syncthreads();
  zline_dft<T, RS>(xl, f, tws, lane);
  if (ok) store_r2c_pair(xl, X + long(nkx) * (2 * p), nkx, nx, lane, f.tpl);
}

// Load of an x c2r row pair into LDS: Z = A + iB from the two half spectra
// (FFTW c2r semantics: Im of kx = 0 and kx = nx/2 ignored), conjugated for the
// backward transform; dirx multiplies both by i kx first.
// KN > 0 (compiled plans, nx <= KN*tpl): every load of the thread is issued
// before the first is used.
template <typename T>
__device__ __forceinline__ cpx<T> c2r_pair_value(cpx<T> A, cpx<T> B, int m, int k, int h,
                                                 int dirx, double kxk) {
  if (dirx) {
    A = ikmul(T(kxk), A);
    B = ikmul(T(kxk), B);
  }
  if (k == 0 || k == h) {
    A.y = 0;
    B.y = 0;
  }
  cpx<T> v = m > h ? mkc<T>(A.x + B.y, -A.y + B.x) : mkc<T>(A.x - B.y, A.y + B.x);
  v.y = -v.y;
  return v;
}

// (the same operations without fused multiply-adds)
template <typename T>
__device__ __forceinline__ cpx<T> c2r_pair_value_nofma(cpx<T> A, cpx<T> B, int m, int k, int h,
                                                       double kxk) {
#pragma clang fp contract(off)
  const T q = T(kxk);
  A = mkc<T>(-(q * A.y), q * A.x);
  B = mkc<T>(-(q * B.y), q * B.x);
  if (k == 0 || k == h) {
    A.y = 0;
    B.y = 0;
  }
  cpx<T> v = m > h ? mkc<T>(A.x + B.y, -A.y + B.x) : mkc<T>(A.x - B.y, A.y + B.x);
  v.y = -v.y;
  return v;
}

// FMA: the derivative's products may be fused into the combination (dirx
// known at compile time); else they are rounded first, whatever the compiler
// does with the branch.
template <typename T, int KN = 0, int CH = KN, bool FMA = true>
__device__ __forceinline__ void load_c2r_pair(cpx<T>* xl, const cpx<T>* __restrict__ a0, int nkx,
                                              int nx, int lane, int tpl, bool ok, int dirx,
                                              const double* __restrict__ kx) {
  const int h = nx / 2;
  if constexpr (KN > 0) {
    // CH elements in flight at a time (CH < KN bounds the registers: the
    // chunk loop stays a loop, so the compiler cannot hoist every load)
#pragma unroll(CH == KN ? KN : 1)
    for (int c0 = 0; c0 < KN; c0 += CH) {
      cpx<T> A[CH], B[CH];
      double kk[CH];
#pragma unroll
      for (int q = 0; q < CH; ++q) {
        const int m = lane + (c0 + q) * tpl;
        const int k = m > h ? nx - m : m;
        A[q] = B[q] = mkc<T>(0, 0);
        kk[q] = 0.0;
        if (ok && m < nx) {
          A[q] = a0[k];
          B[q] = a0[k + nkx];
          if (dirx) kk[q] = kx[k];
        }
      }
#pragma unroll
      for (int q = 0; q < CH; ++q) {
        const int m = lane + (c0 + q) * tpl;
        const int k = m > h ? nx - m : m;
        if (m < nx) {
          cpx<T> v;
          if (!FMA && dirx) v = c2r_pair_value_nofma(A[q], B[q], m, k, h, kk[q]);
          else v = c2r_pair_value(A[q], B[q], m, k, h, FMA ? dirx : 0, kk[q]);
          xl[m] = ok ? v : mkc<T>(0, 0);
        }
      }
    }
  } else {
    for (int m = lane; m < nx; m += tpl) {
      cpx<T> v = mkc<T>(0, 0);
      if (ok) {
        const bool up = m > h;
        const int k = up ? nx - m : m;
        cpx<T> A = a0[k];
        cpx<T> B = a0[k + nkx];
        if (dirx) {
          A = ikmul(T(kx[k]), A);
          B = ikmul(T(kx[k]), B);
        }
        if (k == 0 || k == h) {
          A.y = 0;
          B.y = 0;
        }
        v = up ? mkc<T>(A.x + B.y, -A.y + B.x) : mkc<T>(A.x - B.y, A.y + B.x);
        v.y = -v.y;
      }
      xl[m] = v;
    }
  }
}

template <int RS>
constexpr int batch_n() {
  if constexpr (RS >= RS_WAVE) return keep_n<RS>();
  else return 0;
}
// x lines of a plan whose fused x stage keeps its row pair's velocity in
// registers: powers of two of the general engine (its other radix families
// spill) and the compiled plans of x lines
template <int RS>
constexpr bool xfused_ok() {
  return RS >= RS_WAVE || RS == RS_POW2;
}
template <int RS>
constexpr bool xline_pow2() {
  if constexpr (RS >= RS_WAVE) return (WavePlanOf<RS>::type::m & (WavePlanOf<RS>::type::m - 1)) == 0;
  else return RS == RS_POW2;
}
// whether d/dx in k_xgrad_prod fuses the derivative's product (load_c2r_pair)
template <int RS>
constexpr bool xprod_fma() {
  if constexpr (RS >= RS_WAVE) return WavePlanOf<RS>::type::natural;
  else return false;
}
// The fused x stage holds the velocity of its row pair in registers, so its loads
// are batched in chunks.
template <int RS>
constexpr int xg_chunk() {
  // four elements in flight at a time: at 512^3 the x stage takes 2.2 ms
  // (float32) / 4.2 ms (float64) per RK stage against 2.9 / 5.5 with one
  // and 4.3 / 5.3 with all eight (spills)
  return batch_n<RS>() >= 4 ? 4 : batch_n<RS>();
}

template <typename T, int RS>
__global__ void __launch_bounds__(kMaxBlock) k_xc2r(XFields<T> a, LineFFT<cpx<T>> f, int nkx,
                                              long npairs, int dirx,
                                              const double* __restrict__ kx) {
  using Cp = cpx<T>;
  const Cp* __restrict__ X = static_cast<const Cp*>(a.in[blockIdx.y]);
  T* __restrict__ R = static_cast<T*>(a.out[blockIdx.y]);
  SPX_PROLOGUE(Cp, f);
  const int nx = f.n;
  const long p = long(blockIdx.x) * f.nl + line;
  const bool ok = p < npairs;
  load_c2r_pair<T, batch_n<RS>()>(xl, X + long(nkx) * (2 * (ok ? p : 0)), nkx, nx, lane, f.tpl, ok, dirx, kx);
  __syncthreads();
  zline_dft<T, RS>(xl, f, tws, lane);
  if (ok) {
    T* r0 = R + long(nx) * (2 * p);
    for (int x = lane; x < nx; x += f.tpl) {
      const Cp z = xl[x];
      r0[x] = z.x;
      r0[x + nx] = -z.y;
    }
  }
}

// The x stage of a field's round trip through real space: c2r, ((r/nx)/ny)/nz
// (include/bouss/bouss_rkstep2.f90:57) and r2c of a row pair in LDS, in place on
// its half spectra.  Two field passes instead of the six of k_xc2r, a division
// pass and k_xr2c: 128^3 float64 36 us in three launches, 23 here, bound by the
// three divisions a value.
template <int RS>
__global__ void __launch_bounds__(kMaxBlock) k_xround(cpx<double>* __restrict__ X,
                                                LineFFT<cpx<double>> f, int nkx, long npairs,
                                                double ny, double nz) {
#pragma clang fp contract(off)
  using Cp = cpx<double>;
  SPX_PROLOGUE(Cp, f);
  const int nx = f.n;
  const long p = long(blockIdx.x) * f.nl + line;
  const bool ok = p < npairs;
  Cp* xs = X + long(nkx) * (2 * (ok ? p : 0));
  load_c2r_pair<double, batch_n<RS>()>(xl, xs, nkx, nx, lane, f.tpl, ok, 0, nullptr);
  __syncthreads();
  zline_dft<double, RS>(xl, f, tws, lane);
  for (int x = lane; x < nx; x += f.tpl) {
    const Cp z = xl[x];
    xl[x] = mkc<double>(((z.x / double(nx)) / ny) / nz, ((-z.y / double(nx)) / ny) / nz);
  }
  __syncthreads();
  zline_dft<double, RS>(xl, f, tws, lane);
  if (ok) store_r2c_pair(xl, xs, nkx, nx, lane, f.tpl);
}

// ((u*Dx + v*Dy) + w*Dz)*tmp on a row pair, the three derivatives c2r'd in
// LDS one after the other and accumulated in registers
// (pseudospec_hd.f90:254-312, pseudospec_phd.f90:63-108), then the r2c of the
// product: the real product never goes to memory.  blockIdx.y: field.  The
// half spectra may go over YY: the line that writes a row pair is the one
// that read it.
template <typename T>
struct XProd {
  const cpx<T>* yv[4];
  const cpx<T>* yy[4];
  const cpx<T>* xz[4];
  cpx<T>* out[4];
  const T* vel[3];
};

template <typename T, int RS>
__global__ void __launch_bounds__(kMaxBlock) k_xgrad_prod(XProd<T> a, LineFFT<cpx<T>> f, int nkx,
                                                    long npairs, double tmpd,
                                                    const double* __restrict__ kx) {
#pragma clang fp contract(off)
  using Cp = cpx<T>;
  SPX_PROLOGUE(Cp, f);
  const int nx = f.n;
  const T tmp = T(tmpd);
  const long p = long(blockIdx.x) * f.nl + line;
  const bool ok = p < npairs;
  const long ro = long(nx) * (2 * (ok ? p : 0));
  const long co = long(nkx) * (2 * (ok ? p : 0));
  constexpr int KX = keep_n<RS>();
  T accA[KX], accB[KX];
  const Cp* srcs[3] = {a.yv[blockIdx.y], a.yy[blockIdx.y], a.xz[blockIdx.y]};
  for (int r = 0; r < 3; ++r) {
    if (xprod_fma<RS>() && r == 0)
      load_c2r_pair<T, batch_n<RS>()>(xl, srcs[0] + co, nkx, nx, lane, f.tpl, ok, 1, kx);
    else
      load_c2r_pair<T, batch_n<RS>(), batch_n<RS>(), false>(xl, srcs[r] + co, nkx, nx, lane,
                                                            f.tpl, ok, r == 0 ? 1 : 0, kx);
    // the velocity values this thread multiplies with, loaded before the
    // transform so that their latency overlaps it
    const T* m = a.vel[r] + ro;
    T ma[KX], mb[KX];
#pragma unroll
    for (int q = 0; q < KX; ++q) {
      const int x = lane + q * f.tpl;
      const bool in = x < nx && ok;
      ma[q] = in ? m[x] : T(0);
      mb[q] = in ? m[x + nx] : T(0);
    }
    __syncthreads();
    zline_dft<T, RS>(xl, f, tws, lane);
#pragma unroll
    for (int q = 0; q < KX; ++q) {
      const int x = lane + q * f.tpl;
      if (x < nx) {
        const Cp z = xl[x];
        const T va = z.x, vb = -z.y;
        if (r == 0) {
          accA[q] = ma[q] * va;
          accB[q] = mb[q] * vb;
        } else if (r == 1) {
          accA[q] = accA[q] + ma[q] * va;
          accB[q] = accB[q] + mb[q] * vb;
        } else {
          accA[q] = (accA[q] + ma[q] * va) * tmp;
          accB[q] = (accB[q] + mb[q] * vb) * tmp;
        }
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int q = 0; q < KX; ++q) {
    const int x = lane + q * f.tpl;
    if (x < nx) xl[x] = mkc<T>(accA[q], accB[q]);
  }
  __syncthreads();
  zline_dft<T, RS>(xl, f, tws, lane);
  if (ok) store_r2c_pair(xl, a.out[blockIdx.y] + co, nkx, nx, lane, f.tpl);
}

// gradre's whole x stage on a row pair (pseudospec_hd.f90:254-312): the
// velocity components u, v, w = c2r(YV_c) are formed first and kept in
// registers, then for
// each field c (the three components, and a scalar when nf = 4)
// ((u Dx v_c + v Dy v_c) + w Dz v_c) tmp from the c2r of i kx YV_c, YY_c and
// XZ_c, in k_xgrad_prod's operation order, and its r2c.  Neither the real
// velocity nor the products go to memory.  A line is owned by its tpl threads, so
// the transforms of a row pair synchronise with line_sync.  Launches of fewer
// than kSpread tiles give each field a workgroup of its own (blockIdx.y), which
// forms the velocity again: 7 transforms one after the other instead of 15 (HD
// 32^3 38 -> 20 us, 64^3 45 -> 26 us).
template <typename T>
struct XGradArgs {
  const cpx<T>* yv[4];
  const cpx<T>* yy[4];
  const cpx<T>* xz[4];
  cpx<T>* out[4];
};

template <typename T, int RS>
__global__ void __launch_bounds__(kMaxBlock, sizeof(T) == 4 ? 4 : 2) k_xgrad_fused(
    XGradArgs<T> a, LineFFT<cpx<T>> f, int nkx, long npairs, int nf, double tmpd,
    const double* __restrict__ kx) {
#pragma clang fp contract(off)
  using Cp = cpx<T>;
  SPX_PROLOGUE(Cp, f);
  const int nx = f.n;
  const T tmp = T(tmpd);
  const long p = long(blockIdx.x) * f.nl + line;
  const bool ok = p < npairs;
  const long co = long(nkx) * (2 * (ok ? p : 0));
  constexpr int KX = keep_n<RS>();
  constexpr bool pow2 = xline_pow2<RS>();
  T vel[3][2][KX];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    load_c2r_pair<T, batch_n<RS>(), xg_chunk<RS>()>(xl, a.yv[c] + co, nkx, nx, lane, f.tpl, ok, 0, kx);
    // the first barrier also publishes the staged twiddles
    if (c == 0) __syncthreads();
    else line_sync(f.tpl);
    line_fft_nosync<T, RS>(xl, f, tws, lane);
    line_sync(f.tpl);
#pragma unroll
    for (int q = 0; q < KX; ++q) {
      const int x = lane + q * f.tpl;
      vel[c][0][q] = vel[c][1][q] = T(0);
      if (x < nx) {
        const Cp z = xl[x];
        vel[c][0][q] = z.x;
        vel[c][1][q] = -z.y;
      }
    }
    line_sync(f.tpl);
  }
#pragma unroll 1
  for (int c = blockIdx.y; c < nf; c += gridDim.y) {
    T accA[KX], accB[KX];
    const Cp* srcs[3] = {a.yv[c], a.yy[c], a.xz[c]};
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      // (the scalar's and other lengths' d/dx are k_xgrad_prod's to the bit)
      if (r == 0 && (!pow2 || c == 3))
        load_c2r_pair<T, batch_n<RS>(), xg_chunk<RS>(), false>(
            xl, srcs[r] + co, nkx, nx, lane, f.tpl, ok, 1, kx);
      else
        load_c2r_pair<T, batch_n<RS>(), xg_chunk<RS>()>(xl, srcs[r] + co, nkx, nx, lane,
                                                              f.tpl, ok, r == 0 ? 1 : 0, kx);
      line_sync(f.tpl);
      line_fft_nosync<T, RS>(xl, f, tws, lane);
      line_sync(f.tpl);
#pragma unroll
      for (int q = 0; q < KX; ++q) {
        const int x = lane + q * f.tpl;
        if (x < nx) {
          const Cp z = xl[x];
          const T va = z.x, vb = -z.y;
          if (r == 0) {
            accA[q] = vel[0][0][q] * va;
            accB[q] = vel[0][1][q] * vb;
          } else if (r == 1) {
            accA[q] = accA[q] + vel[1][0][q] * va;
            accB[q] = accB[q] + vel[1][1][q] * vb;
          } else {
            // the element's own thread read it: the product replaces it
            xl[x] = mkc<T>((accA[q] + vel[2][0][q] * va) * tmp,
                           (accB[q] + vel[2][1][q] * vb) * tmp);
          }
        }
      }
      line_sync(f.tpl);
    }
    line_fft_nosync<T, RS>(xl, f, tws, lane);
    line_sync(f.tpl);
    if (ok) store_r2c_pair(xl, a.out[c] + co, nkx, nx, lane, f.tpl);
    line_sync(f.tpl);
  }
}

using Cd = cpx<double>;
// The x stage of a cross product A x B on a row pair (pseudospec_hd.f90:383-399,
// pseudospec_mhd.f90 vector): the c2r of A's components, kept in registers,
// then of B's one after the other with the partial products they enter, and the
// r2c of the three results; neither the real fields nor the products go to
// memory.  k_xc2r, k_cross_real and k_xr2c moved 69 field passes for the three
// products of a stage (128^3, two stages: 460 us), this kernel 27 (277 us; one to
// two waves per SIMD at 190 to 256 registers, 3.3 TB/s).  out may be
// A's or B's buffers: the line that writes a row pair is the one that read it.
struct XCross {
  const cpx<double>* a[3];
  const cpx<double>* b[3];
  cpx<double>* out[3];
};
// five of the six components' values live at a time: up to 8 points per lane
// stay within two waves per SIMD's registers
template <int RS>
constexpr bool xcross_ok() {
  if constexpr (RS >= RS_WAVE) return keep_n<RS>() <= 8;
  else return false;
}

template <int RS>
__global__ void __launch_bounds__(kMaxBlock, 2) k_xcross(XCross a, LineFFT<Cd> f, int nkx,
                                                   long npairs, double tmp) {
#pragma clang fp contract(off)
  SPX_PROLOGUE(Cd, f);
  const int nx = f.n;
  const long p = long(blockIdx.x) * f.nl + line;
  const bool ok = p < npairs;
  const long co = long(nkx) * (2 * (ok ? p : 0));
  constexpr int KX = keep_n<RS>(), CH = KX >= 4 ? 4 : KX;
  double A[3][2][KX], P1[2][KX], P2[2][KX], P3[2][KX];
  // values of one field: use(q, row, value)
  auto field = [&](const Cd* src, bool first, auto use) {
    load_c2r_pair<double, KX, CH>(xl, src + co, nkx, nx, lane, f.tpl, ok, 0, nullptr);
    if (first) __syncthreads();  // also publishes the staged twiddles
    else line_sync(f.tpl);
    line_fft_nosync<double, RS>(xl, f, tws, lane);
    line_sync(f.tpl);
#pragma unroll
    for (int q = 0; q < KX; ++q) {
      const int x = lane + q * f.tpl;
      const Cd z = x < nx ? xl[x] : mkc<double>(0, 0);
      use(q, 0, z.x);
      use(q, 1, -z.y);
    }
    line_sync(f.tpl);
  };
#pragma unroll
  for (int c = 0; c < 3; ++c)
    field(a.a[c], c == 0, [&](int q, int r, double v) { A[c][r][q] = v; });
  field(a.b[0], false, [&](int q, int r, double v) {
    P2[r][q] = A[2][r][q] * v;
    P3[r][q] = v * A[1][r][q];
  });
  field(a.b[1], false, [&](int q, int r, double v) {
    P1[r][q] = v * A[2][r][q];
    P3[r][q] = (A[0][r][q] * v - P3[r][q]) * tmp;
  });
  field(a.b[2], false, [&](int q, int r, double v) {
    P1[r][q] = (A[1][r][q] * v - P1[r][q]) * tmp;
    P2[r][q] = (P2[r][q] - v * A[0][r][q]) * tmp;
  });
  auto result = [&](Cd* out, const double (&o)[2][KX]) {
#pragma unroll
    for (int q = 0; q < KX; ++q) {
      const int x = lane + q * f.tpl;
      if (x < nx) xl[x] = ok ? mkc<double>(o[0][q], o[1][q]) : mkc<double>(0, 0);
    }
    line_sync(f.tpl);
    line_fft_nosync<double, RS>(xl, f, tws, lane);
    line_sync(f.tpl);
    if (ok) store_r2c_pair(xl, out + co, nkx, nx, lane, f.tpl);
    line_sync(f.tpl);
  };
  result(a.out[0], P1);
  result(a.out[1], P2);
  result(a.out[2], P3);
}

// ---------------------------------------------------------------------------
// float64 boundary kernels; TS is the storage type of the fields
// ---------------------------------------------------------------------------
using LFd = LineFFT<Cd>;

// goto_domain_w_boundaries + noslip_z + goto_3d_fourier fused per line
// (boundary_mod.fpp:72-194, vboundary.f90:154-211, sboundary.f90:122-165).
// comp 0: vx (kx), comp 1: vy (ky); scalar mode: wall values are zero.

template <typename TS, int RS>
__global__ void __launch_bounds__(kMaxBlock) k_noslip(cpx<TS>* __restrict__ vx, cpx<TS>* __restrict__ vy,
                                                const Cd* __restrict__ pr, LFd f, long nlines,
                                                int ny, int np, double invn, WallParams wp,
                                                const double* __restrict__ kx,
                                                const double* __restrict__ ky,
                                                const double* __restrict__ dir, int C, int d,
                                                RkLoad rk, int rk_on) {
#pragma clang fp contract(off)
  SPX_PROLOGUE(Cd, f);
  const int n = f.n;
  const int comp = blockIdx.y;
  cpx<TS>* V = comp ? vy : vx;
  const long ln = long(blockIdx.x) * f.nl + line;
  const bool ok = ln < nlines;
  const long li = ok ? ln / ny : 0;
  const int lj = ok ? int(ln - li * ny) : 0;
  // wall value of lanes 0 (z = 0) and 1 (z = Lz), read before the transform
  Cd val = mkc<double>(0, 0);
  if (lane < 2 && ok && !wp.scalar) {
    const int ind = lane ? np - 1 : 0;
    const Cd pv = pr[ln * n + ind];
    const double kxi = kx[li], kyj = ky[lj];
    val = cscale(ikmul(comp ? kyj : kxi, pv), wp.tau);
    if (kxi == 0.0 && kyj == 0.0) val = mkc<double>(wp.nxny * wp.vb[comp][lane], 0.0);
  }
  for (int k = lane; k < n; k += f.tpl) {
    Cd v = mkc<double>(0, 0);
    if (ok) {
      v = ccast<double>(V[ln * n + k]);
      if (rk_on) v = rk_on_load(rk, comp, v, ln * n + k, li, lj, k);
    }
    xl[k] = cconj(v);
  }
  __syncthreads();
  line_dft<double, RS>(xl, f, tws, lane);
  for (int k = lane; k < np; k += f.tpl) xl[k] = cscale(cconj(xl[k]), invn);
  __syncthreads();
  if (lane < 2 && ok) xl[lane ? np - 1 : 0] = val;
  __syncthreads();
  fc_continue_lds(lds, f.nl, f.ldl, np, C, d, dir);
  __syncthreads();
  line_dft<double, RS>(xl, f, tws, lane);
  if (ok)
    for (int k = lane; k < n; k += f.tpl) V[ln * n + k] = ccast<TS>(xl[k]);
}

// goto_domain_w_boundaries + the magnetic wall conditions + goto_3d_fourier
// fused per line (boundary_mod.fpp:72-194, bboundary.f90:192-344,
// fcgram_mod.f90:437-468, 550-568); blockIdx.y = component (a0, a1, a2).
template <typename TS, int RS>
__global__ void __launch_bounds__(kMaxBlock) k_bwall(Cd* __restrict__ a0, Cd* __restrict__ a1,
                                                     Cd* __restrict__ a2, LFd f, long nlines,
                                                     int np, double invn, BWallParams bp,
                                                     const double* __restrict__ khom,
                                                     const double* __restrict__ dir, int C,
                                                     int d) {
#pragma clang fp contract(off)
  SPX_PROLOGUE(Cd, f);
  const int n = f.n;
  const int comp = blockIdx.y;
  Cd* V = comp == 0 ? a0 : (comp == 1 ? a1 : a2);
  const long ln = long(blockIdx.x) * f.nl + line;
  const bool ok = ln < nlines;
  for (int k = lane; k < n; k += f.tpl) xl[k] = ok ? cconj(V[ln * n + k]) : mkc<double>(0, 0);
  __syncthreads();
  zline_dft<double, RS>(xl, f, tws, lane);
  for (int k = lane; k < np; k += f.tpl) xl[k] = cscale(cconj(xl[k]), invn);
  __syncthreads();
  // lane 0: the wall at z = 0, lane 1: z = Lz (their stencils do not overlap
  // for np > d)
  if (lane < 2 && ok) {
    const int m = bp.mode[comp][lane];
    if (m) {
      const int ind = lane ? np - 1 : 0;
      xl[ind] = mkc<double>(0, 0);
      if (m >= 2) {
        const double* vec = m == 3 ? bp.neu2 : bp.neu1;
        Cd acc = cscale(xl[ind], vec[d - 1]);
        for (int k = 0; k < d - 1; ++k)
          acc = cadd(acc, cscale(xl[lane ? np - d + k : d - 1 - k], vec[k]));
        if (m == 4) {
          const double den = khom[ln] * vec[d - 1] + 1;
          acc = mkc<double>(acc.x / den, acc.y / den);
        }
        xl[ind] = acc;
      }
    }
  }
  __syncthreads();
  fc_continue_lds(lds, f.nl, f.ldl, np, C, d, dir);
  __syncthreads();
  zline_dft<double, RS>(xl, f, tws, lane);
  if (ok)
    for (int k = lane; k < n; k += f.tpl) V[ln * n + k] = xl[k];
}

// laplace_z pure-Neumann coefficients (boundary_mod.fpp:531-560)
struct Coef {
  Cd c1, c2;
};
__device__ __forceinline__ Coef neumann_coef(Cd b1, Cd b2, double kh, double Lz, bool zero_mode) {
#pragma clang fp contract(off)
  Coef r;
  if (zero_mode) {
    r.c1 = b1;
    r.c2 = mkc<double>(0, 0);
    return r;
  }
  const double tmp = 1.0 / (kh * (1 - exp(-2 * kh * Lz)));
  const double e1 = exp(-kh * Lz);
  r.c1 = cscale(csub(b2, cscale(b1, e1)), tmp);
  r.c2 = cscale(cadd(mkc<double>(-b1.x, -b1.y), cscale(b2, e1)), tmp);
  return r;
}

// laplace_z coefficients for the wall kinds (k0, k1) (boundary_mod.fpp:497-621):
// 0 Dirichlet, 1 Neumann, 2 Robin with constant khom; (1,1), (0,0), (2,2), (0,2)
__device__ __forceinline__ Coef laplace_coef(int k0, int k1, Cd b1, Cd b2, double kh, double Lz,
                                             bool zero_mode) {
#pragma clang fp contract(off)
  if (k0 == 1) return neumann_coef(b1, b2, kh, Lz, zero_mode);
  Coef r;
  if (k0 == 0 && k1 == 0) {
    if (zero_mode) {
      const Cd t = csub(b2, b1);
      r.c1 = mkc<double>(t.x / Lz, t.y / Lz);
      r.c2 = b1;
      return r;
    }
    const double tmp = 1.0 / (1 - exp(-2 * kh * Lz));
    const double e1 = exp(-kh * Lz);
    r.c1 = cscale(csub(b2, cscale(b1, e1)), tmp);
    r.c2 = cscale(csub(b1, cscale(b2, e1)), tmp);
    return r;
  }
  if (k0 == 2) {  // (2,2)
    if (zero_mode) {
      r.c1 = b1;
      r.c2 = mkc<double>(0, 0);
      return r;
    }
    const double tmp = 1.0 / (2 * kh);
    r.c1 = cscale(b2, tmp);
    r.c2 = cscale(b1, tmp);
    return r;
  }
  // (0,2)
  if (zero_mode) {
    r.c1 = b2;
    r.c2 = b1;
    return r;
  }
  const double tmp = 1.0 / (2 * kh);
  r.c1 = cscale(b2, tmp);
  r.c2 = cscale(csub(cscale(cscale(b1, 2.0), kh), cscale(b2, exp(-kh * Lz))), tmp);
  return r;
}

// d <- IFFT_z(d)*tmp + a_harm(z)  (:354-381 with laplace_z :631-675); d is float64
// (TS = double: the kernels of this family are instantiated per type)
template <typename TS, int RS>
__global__ void __launch_bounds__(kMaxBlock) k_proj_pressure(Cd* __restrict__ dd,
                                                       const Cd* __restrict__ bc, LFd f,
                                                       long nlines, int ny, double tmp, double Lz,
                                                       const double* __restrict__ khom,
                                                       const double* __restrict__ z, int k0,
                                                       int k1) {
#pragma clang fp contract(off)
  SPX_PROLOGUE(Cd, f);
  const int n = f.n;
  const long ln = long(blockIdx.x) * f.nl + line;
  const bool ok = ln < nlines;
  if constexpr (RS >= RS_WAVE) {
    constexpr int KN = keep_n<RS>();
    Cd v[KN];
#pragma unroll
    for (int q = 0; q < KN; ++q) {
      const int k = lane + q * f.tpl;
      v[q] = mkc<double>(0, 0);
      if (ok && k < n) v[q] = cconj(dd[ln * n + k]);
    }
#pragma unroll
    for (int q = 0; q < KN; ++q) {
      const int k = lane + q * f.tpl;
      if (k < n) xl[k] = v[q];
    }
  } else {
    for (int k = lane; k < n; k += f.tpl) xl[k] = ok ? cconj(dd[ln * n + k]) : mkc<double>(0, 0);
  }
  // (kx, ky) = (0, 0) is the only line with khom = 0; coefficients formed
  // before the transform
  const double kh = ok ? khom[ln] : 1.0;
  const bool zm = kh == 0.0;
  Coef cf;
  cf.c1 = cf.c2 = mkc<double>(0, 0);
  if (ok) cf = laplace_coef(k0, k1, bc[2 * ln], bc[2 * ln + 1], kh, Lz, zm);
  __syncthreads();
  zline_dft<double, RS>(xl, f, tws, lane);
  if (!ok) return;
  for (int k = lane; k < n; k += f.tpl) {
    Cd a;
    if (zm) {
      a = mkc<double>(cf.c1.x * z[k] + cf.c2.x, 0.0);
    } else {
      const double ep = exp(kh * (z[k] - Lz));
      const double em = exp(-kh * z[k]);
      a = cadd(cscale(cf.c1, ep), cscale(cf.c2, em));
    }
    dd[ln * n + k] = cadd(cscale(cconj(xl[k]), tmp), a);
  }
}

// k_proj_pressure at z = 0 and z = np-1 only, one thread per line, from the
// wall values pw = IFFT_z(d)/nz formed by the projection kernel
static __global__ void k_pressure_walls(Cd* __restrict__ dd, const Cd* __restrict__ bc,
                                 const Cd* __restrict__ pw, long nlines, int n, int np,
                                 double Lz, const double* __restrict__ khom,
                                 const double* __restrict__ z) {
#pragma clang fp contract(off)
  const long ln = long(blockIdx.x) * blockDim.x + threadIdx.x;
  if (ln >= nlines) return;
  const double kh = khom[ln];
  const bool zm = kh == 0.0;
  const Coef cf = neumann_coef(bc[2 * ln], bc[2 * ln + 1], kh, Lz, zm);
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    const int k = w ? np - 1 : 0;
    Cd a;
    if (zm) {
      a = mkc<double>(cf.c1.x * z[k] + cf.c2.x, 0.0);
    } else {
      const double ep = exp(kh * (z[k] - Lz));
      const double em = exp(-kh * z[k]);
      a = cadd(cscale(cf.c1, ep), cscale(cf.c2, em));
    }
    dd[ln * n + k] = cadd(pw[2 * ln + w], a);
  }
}

// harmonic correction: A = FFT_z(cont(a_harm)), B = FFT_z(cont(d a_harm/dz));
// vx -= i kx A, vy -= i ky A, vz -= B   (:383-399).  Two buffers per line.
template <typename TS, int RS>
__global__ void __launch_bounds__(kMaxBlock) k_proj_harmonic(cpx<TS>* __restrict__ va,
                                                       cpx<TS>* __restrict__ vb,
                                                       cpx<TS>* __restrict__ vc,
                                                       const Cd* __restrict__ bc, LFd f,
                                                       long nlines, int ny, int np, double Lz,
                                                       const double* __restrict__ khom,
                                                       const double* __restrict__ z,
                                                       const double* __restrict__ kx,
                                                       const double* __restrict__ ky,
                                                       const double* __restrict__ dir, int C,
                                                       int d, int k0, int k1) {
#pragma clang fp contract(off)
  SPX_PROLOGUE(Cd, f);
  const int n = f.n;
  Cd* const ldsB = lds + f.nl * f.ldl;
  Cd* const xb = ldsB + line * f.ldl;
  const long ln = long(blockIdx.x) * f.nl + line;
  const bool ok = ln < nlines;
  const long i = ok ? ln / ny : 0;
  const int j = ok ? int(ln - i * ny) : 0;
  const double kh = ok ? khom[ln] : 0.0;
  const bool zm = kh == 0.0;
  Coef cf;
  cf.c1 = cf.c2 = mkc<double>(0, 0);
  if (ok) cf = laplace_coef(k0, k1, bc[2 * ln], bc[2 * ln + 1], kh, Lz, zm);
  // the field values this thread corrects, read before the transforms (the
  // two line buffers bound the occupancy, not the registers)
  Cd pa[KEEP], pb[KEEP], pc[KEEP];
#pragma unroll
  for (int q = 0; q < KEEP; ++q) {
    const int k = lane + q * f.tpl;
    if (ok && k < n) {
      const long o = ln * n + k;
      pa[q] = ccast<double>(va[o]);
      pb[q] = ccast<double>(vb[o]);
      pc[q] = ccast<double>(vc[o]);
    }
  }
  for (int k = lane; k < np; k += f.tpl) {
    Cd a = mkc<double>(0, 0), b = mkc<double>(0, 0);
    if (ok) {
      if (zm) {
        a = mkc<double>(cf.c1.x * z[k] + cf.c2.x, 0.0);
        b = mkc<double>(cf.c1.x, 0.0);
      } else {
        const double ep = exp(kh * (z[k] - Lz));
        const double em = exp(-kh * z[k]);
        const Cd t1 = cscale(cf.c1, ep), t2 = cscale(cf.c2, em);
        a = cadd(t1, t2);
        b = cscale(csub(t1, t2), kh);
      }
    }
    xl[k] = a;
    xb[k] = b;
  }
  __syncthreads();
  fc_continue_lds(lds, f.nl, f.ldl, np, C, d, dir);
  fc_continue_lds(ldsB, f.nl, f.ldl, np, C, d, dir);
  __syncthreads();
  line_dft<double, RS>(xl, f, tws, lane);
  line_dft<double, RS>(xb, f, tws, lane);
  if (!ok) return;
  const double kxi = kx[i], kyj = ky[j];
#pragma unroll
  for (int q = 0; q < KEEP; ++q) {
    const int k = lane + q * f.tpl;
    if (k < n) {
      const Cd A = xl[k], B = xb[k];
      const long o = ln * n + k;
      va[o] = ccast<TS>(csub(pa[q], ikmul(kxi, A)));
      vb[o] = ccast<TS>(csub(pb[q], ikmul(kyj, A)));
      vc[o] = ccast<TS>(csub(pc[q], B));
    }
  }
}

// The two harmonic profiles of each distinct khom value u on the physical
// points, rows 2u and 2u+1 of tab (continued and transformed afterwards).
static __global__ void k_harm_profiles(Cd* __restrict__ tab, const double* __restrict__ khv, int U,
                                int n, int np, const double* __restrict__ z, double Lz) {
#pragma clang fp contract(off)
  const long e = long(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= long(U) * np) return;
  const int u = int(e / np), k = int(e - long(u) * np);
  const double kh = khv[u];
  double a1, a2;
  if (kh == 0.0) {
    a1 = z[k];
    a2 = 1.0;
  } else {
    a1 = exp(kh * (z[k] - Lz));
    a2 = exp(-kh * z[k]);
  }
  tab[(2 * long(u)) * n + k] = mkc<double>(a1, 0.0);
  tab[(2 * long(u) + 1) * n + k] = mkc<double>(a2, 0.0);
}

// Harmonic correction from the basis table, one wavefront per line:
// A = c1 P1 + c2 P2, B = kh (c1 P1 - c2 P2) (kh = 0: A = Re c1 P1 + Re c2 P2,
// B = Re c1 P2); vx -= i kx A, vy -= i ky A, vz -= B   (:383-399).
template <typename TS>
__global__ void __launch_bounds__(256) k_proj_harmonic_tab(cpx<TS>* __restrict__ va,
                                                         cpx<TS>* __restrict__ vb,
                                                         cpx<TS>* __restrict__ vc,
                                                         const Cd* __restrict__ bc,
                                                         const Cd* __restrict__ tab,
                                                         const int* __restrict__ hidx,
                                                         long nlines, int ny, int n, double Lz,
                                                         const double* __restrict__ khom,
                                                         const double* __restrict__ kx,
                                                         const double* __restrict__ ky, int k0,
                                                         int k1) {
#pragma clang fp contract(off)
  const long ln = long(blockIdx.x) * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (ln >= nlines) return;
  const long i = ln / ny;
  const int j = int(ln - i * ny);
  const double kh = khom[ln];
  const bool zm = kh == 0.0;
  const Coef cf = laplace_coef(k0, k1, bc[2 * ln], bc[2 * ln + 1], kh, Lz, zm);
  const Cd* P1 = tab + 2 * long(hidx[ln]) * n;
  const Cd* P2 = P1 + n;
  const double kxi = kx[i], kyj = ky[j];
  for (int k = lane; k < n; k += 64) {
    const Cd p1 = P1[k], p2 = P2[k];
    Cd A, B;
    if (zm) {
      A = cadd(cscale(p1, cf.c1.x), cscale(p2, cf.c2.x));
      B = cscale(p2, cf.c1.x);
    } else {
      const Cd u1 = cmul(cf.c1, p1), u2 = cmul(cf.c2, p2);
      A = cadd(u1, u2);
      B = cscale(csub(u1, u2), kh);
    }
    const long o = ln * n + k;
    va[o] = ccast<TS>(csub(ccast<double>(va[o]), ikmul(kxi, A)));
    vb[o] = ccast<TS>(csub(ccast<double>(vb[o]), ikmul(kyj, A)));
    vc[o] = ccast<TS>(csub(ccast<double>(vc[o]), B));
  }
}

// sol_project in one pass per line (boundary_mod.fpp:197-402 with
// poisson_inhomogeneous :405-448 and laplace_z :451-678), one wavefront per
// (kx, ky) line holding its KPL points per lane in registers:
//   d = -i(kx a + ky b + kz c)/kz2 (d(0,0,0) = 0), v -= i k d   (first projection)
//   bc = IFFT_z(c/nz) at z = 0 and z = Lz as two DFT sums        (wall data)
//   A = c1 P1 + c2 P2, B = kh (c1 P1 - c2 P2) from bc and the    (harmonic correction
//   basis table; v -= (i kx A, i ky A, B)                           from the table)
// The arithmetic of every value is that of k_poisson_project_bc followed by
// k_proj_harmonic_tab; the projected velocity never goes through HBM.
// vz takes the RK update on its load when rk_on; pw (when non-null) gets
// IFFT_z(d)/nz at the two walls and d is then not written there.
// RKM < 0: any nz, RK update chosen at run time (rk_on); RKM >= 0: nz >=
// 64 (KPL - 1), so that only the last of a lane's points can lie past the line
// end and the others are loaded without a branch between them; RKM 0: no RK
// update, 1: RK update with a float64 nonlinear term, 2: float32.  Register
// budget of the branch-free forms: 2 waves per SIMD up to 9 points per lane
// (HD 512^3: 2.43 ms per launch against 2.81 at one wave), one wave for 17
// (HD 1024^3: 23.1 ms against 25.8 for the general form).
template <int KPL, int RKM>
__global__ void __launch_bounds__(256, RKM >= 0 && KPL <= 9 ? 2 : 1) k_project_harmonic(
    Cd* __restrict__ a, Cd* __restrict__ b, Cd* __restrict__ c, Cd* __restrict__ d,
    Cd* __restrict__ bc, long nlines, int nz, int ny, const double* __restrict__ kx,
    const double* __restrict__ ky, const double* __restrict__ kz, const Cd* __restrict__ wtop,
    double tmp, RkLoad rk, int rk_on, Cd* __restrict__ pw, int np, const Cd* __restrict__ tab,
    const int* __restrict__ hidx, double Lz, const double* __restrict__ khom) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const long ln = long(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (ln >= nlines) return;  // uniform per wavefront
  const long i = ln / ny;
  const int j = int(ln - i * ny);
  const double kxi = kx[i], kyj = ky[j];
  // the RK update's factors of the line (rk_on_load's, read once)
  double rkl2 = 0.0, rfx = 0.0, rfy = 0.0, rnu = 0.0;
  if constexpr (RKM > 0) {
    const double rx = rk.kx[i], ry = rk.ky[j];
    rkl2 = rx * rx + ry * ry;
    rfx = rk.fkx[i];
    rfy = rk.fky[j];
    rnu = rk.c[0].nu[i];
  }
  Cd s0 = mkc<double>(0, 0), s1 = mkc<double>(0, 0);
  Cd q0 = mkc<double>(0, 0), q1 = mkc<double>(0, 0);
  Cd pa[KPL], pb[KPL], pc[KPL];
#pragma unroll
  for (int q = 0; q < KPL; ++q) {
    const int k = lane + 64 * q;
    if ((RKM >= 0 && q < KPL - 1) || k < nz) {
      const long e = ln * nz + k;
      const double kzk = kz[k];
      const double kk2 = (kxi * kxi + kyj * kyj) + kzk * kzk;
      const Cd A = a[e], B = b[e];
      Cd Cc = c[e];
      if constexpr (RKM < 0) {
        if (rk_on) Cc = rk_on_load(rk, 0, Cc, e, i, j, k);
      } else if constexpr (RKM > 0) {
        Cd nl;
        if constexpr (RKM == 2) {
          const cpx<float> t = static_cast<const cpx<float>*>(rk.c[0].nl)[e];
          nl = mkc<double>(double(t.x), double(t.y));
        } else {
          nl = static_cast<const Cd*>(rk.c[0].nl)[e];
        }
        Cc = rk_apply(rk, Cc, nl, static_cast<const Cd*>(rk.c[0].f)[e],
                      static_cast<const Cd*>(rk.c[0].c0)[e], rkl2, rk.kz[k], rfx, rfy, rk.fkz[k],
                      rnu);
      }
      Cd sm = cadd(cscale(A, kxi), cscale(B, kyj));
      sm = cadd(sm, cscale(Cc, kzk));
      Cd dd;
      if (kk2 == 0.0) {  // the (0,0,0) mode
        dd = mkc<double>(0, 0);
      } else {
        dd = mkc<double>(sm.y / kk2, -sm.x / kk2);
      }
      if (pw) {
        q0 = cadd(q0, dd);
        q1 = cadd(q1, cmul(dd, wtop[k]));
        if (k != 0 && k != np - 1) d[e] = dd;
      } else {
        d[e] = dd;
      }
      pa[q] = csub(A, ikmul(kxi, dd));
      pb[q] = csub(B, ikmul(kyj, dd));
      pc[q] = csub(Cc, ikmul(kzk, dd));
      const Cd c1 = cscale(pc[q], tmp);
      s0 = cadd(s0, c1);
      s1 = cadd(s1, cmul(c1, wtop[k]));
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    s0.x += __shfl_xor(s0.x, off);
    s0.y += __shfl_xor(s0.y, off);
    s1.x += __shfl_xor(s1.x, off);
    s1.y += __shfl_xor(s1.y, off);
  }
  if (lane == 0) {
    bc[2 * ln] = s0;
    bc[2 * ln + 1] = s1;
  }
  if (pw) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      q0.x += __shfl_xor(q0.x, off);
      q0.y += __shfl_xor(q0.y, off);
      q1.x += __shfl_xor(q1.x, off);
      q1.y += __shfl_xor(q1.y, off);
    }
    if (lane == 0) {
      pw[2 * ln] = cscale(q0, tmp);
      pw[2 * ln + 1] = cscale(q1, tmp);
    }
  }
  // harmonic correction (the k_proj_harmonic_tab arithmetic)
  const double kh = khom[ln];
  const bool zm = kh == 0.0;
  const Coef cf = neumann_coef(s0, s1, kh, Lz, zm);
  const Cd* P1 = tab + 2 * long(hidx[ln]) * nz;
  const Cd* P2 = P1 + nz;
#pragma unroll
  for (int q = 0; q < KPL; ++q) {
    const int k = lane + 64 * q;
    if ((RKM >= 0 && q < KPL - 1) || k < nz) {
      const Cd p1 = P1[k], p2 = P2[k];
      Cd A, B;
      if (zm) {
        A = cadd(cscale(p1, cf.c1.x), cscale(p2, cf.c2.x));
        B = cscale(p2, cf.c1.x);
      } else {
        const Cd u1 = cmul(cf.c1, p1), u2 = cmul(cf.c2, p2);
        A = cadd(u1, u2);
        B = cscale(csub(u1, u2), kh);
      }
      const long o = ln * nz + k;
      a[o] = csub(pa[q], ikmul(kxi, A));
      b[o] = csub(pb[q], ikmul(kyj, A));
      c[o] = csub(pc[q], B);
    }
  }
}

// ---------------------------------------------------------------------------
// diagnostics: per-line float64 reductions over physical z in the mixed domain
// ---------------------------------------------------------------------------
__device__ __forceinline__ double line_reduce(double v, double* red, int line, int lane, int tpl) {
  red[line * tpl + lane] = v;
  __syncthreads();
  for (int s = tpl >> 1; s > 0; s >>= 1) {
    if (lane < s) red[line * tpl + lane] += red[line * tpl + lane + s];
    __syncthreads();
  }
  return red[line * tpl];
}

template <typename TS>
struct LinCombDev {
  const cpx<TS>* in[3];
  int dir[3];
  int sgn[3];
};

// dirn 1..3: (i k_dirn) v ; 4: kk2 v with kk2 = (kx^2 + ky^2) + kz^2
__device__ __forceinline__ Cd deriv_apply(Cd v, int dirn, double kxi, double kyj, double kzk) {
#pragma clang fp contract(off)
  if (dirn == 1) return ikmul(kxi, v);
  if (dirn == 2) return ikmul(kyj, v);
  if (dirn == 3) return ikmul(kzk, v);
  if (dirn == 4) return cscale(v, (kxi * kxi + kyj * kyj) + kzk * kzk);
  return v;
}

// The terms of one diagnostic (blockIdx.y): a field or combination each, with
// its factor field of mode 1.
template <typename TS>
struct ZTerms {
  LinCombDev<TS> lc[3];
  const cpx<TS>* b[3];
};

// mode 0: sum_k<np |IFFT(lincomb)|^2 ; mode 1: Re(IFFT(a) conj IFFT(b)) ; mode 2: walls |.|^2 ;
// mode 3: the wall values IFFT(lincomb) at z = 0 and z = Lz (4 doubles per line).
// Term t writes its lines' values at out + t nlines (1, 2 or 4 doubles).
template <typename TS, int RS>
__global__ void __launch_bounds__(kMaxBlock) k_zline_reduce(ZTerms<TS> terms, int mode,
                                                      double* __restrict__ outs, LFd f,
                                                      long nlines, int ny, int np,
                                                      const double* __restrict__ kx,
                                                      const double* __restrict__ ky,
                                                      const double* __restrict__ kz) {
#pragma clang fp contract(off)
  const LinCombDev<TS> lc = terms.lc[blockIdx.y];
  const cpx<TS>* __restrict__ bsrc = terms.b[blockIdx.y];
  SPX_PROLOGUE(Cd, f);
  const int n = f.n;
  double* __restrict__ out = outs + blockIdx.y * nlines * (mode == 3 ? 4 : (mode == 2 ? 2 : 1));
  Cd* const ldsB = lds + f.nl * f.ldl;
  Cd* const xb = ldsB + line * f.ldl;
  double* red = reinterpret_cast<double*>(ldsB + (mode == 1 ? f.nl * f.ldl : 0));
  const long ln = long(blockIdx.x) * f.nl + line;
  const bool ok = ln < nlines;
  const long i = ok ? ln / ny : 0;
  const int j = ok ? int(ln - i * ny) : 0;
  for (int k = lane; k < n; k += f.tpl) {
    Cd v = mkc<double>(0, 0), w = mkc<double>(0, 0);
    if (ok) {
      const double kxi = kx[i], kyj = ky[j], kzk = kz[k];
      v = deriv_apply(ccast<double>(lc.in[0][ln * n + k]), lc.dir[0], kxi, kyj, kzk);
#pragma unroll
      for (int t = 1; t < 3; ++t) {
        if (lc.sgn[t] == 0) continue;
        const Cd u = deriv_apply(ccast<double>(lc.in[t][ln * n + k]), lc.dir[t], kxi, kyj, kzk);
        v = lc.sgn[t] > 0 ? cadd(v, u) : csub(v, u);
      }
      if (mode == 1) w = ccast<double>(bsrc[ln * n + k]);
    }
    xl[k] = cconj(v);
    if (mode == 1) xb[k] = cconj(w);
  }
  __syncthreads();
  zline_dft<double, RS>(xl, f, tws, lane);
  if (mode == 1) zline_dft<double, RS>(xb, f, tws, lane);
  if (mode == 2) {
    if (lane == 0 && ok) {
      const Cd b = xl[0], t = xl[np - 1];
      out[2 * ln] = b.x * b.x + b.y * b.y;
      out[2 * ln + 1] = t.x * t.x + t.y * t.y;
    }
    return;
  }
  if (mode == 3) {
    // the line holds conj(IFFT)
    if (lane == 0 && ok) {
      const Cd b = xl[0], t = xl[np - 1];
      out[4 * ln] = b.x;
      out[4 * ln + 1] = -b.y;
      out[4 * ln + 2] = t.x;
      out[4 * ln + 3] = -t.y;
    }
    return;
  }
  double acc = 0.0;
  for (int k = lane; k < np; k += f.tpl) {
    const Cd v = xl[k];
    if (mode == 0) {
      acc += v.x * v.x + v.y * v.y;
    } else {
      const Cd w = xb[k];
      // values hold conj(IFFT); Re(p conj(q)) is invariant under conj of both
      acc += v.x * w.x + v.y * w.y;
    }
  }
  const double s = line_reduce(acc, red, line, lane, f.tpl);
  if (lane == 0 && ok) out[ln] = s;
}

#if !defined(SPX_PART) || SPX_PART == 8
// The sum over a member's (kx, ky) lines of the weighted terms, lines of kx > 0
// counted twice: blockIdx.x member, blockIdx.y which of the line's per values.
// In a fixed order: a thread's lines upwards, then a tree over the threads.
struct LineWeights {
  double w[3];
};
__global__ void __launch_bounds__(1024) k_line_sum(const double* __restrict__ part, LineWeights w,
                                             int nterm, int per, long nl, int ny,
                                             double* __restrict__ out) {
#pragma clang fp contract(off)
  __shared__ double red[1024];
  const long lines = nl * gridDim.x, l0 = nl * blockIdx.x;
  double s = 0.0;
  for (long l = threadIdx.x; l < nl; l += 1024) {
    double a = 0.0;
    for (int t = 0; t < nterm; ++t)
      a += w.w[t] * part[(t * lines + l0 + l) * per + blockIdx.y];
    s += l < ny ? a : 2.0 * a;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int q = 512; q > 0; q >>= 1) {
    if (threadIdx.x < q) red[threadIdx.x] += red[threadIdx.x + q];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.y * gridDim.x + blockIdx.x] = red[0];
}
#endif

#if !defined(SPX_PART) || SPX_PART == 1
// ---------------------------------------------------------------------------
// plan construction: algorithm choice, factorisation, long-double tables
// ---------------------------------------------------------------------------
static bool factor_small(int n, std::vector<int>& fac) {
  fac.clear();
  int a = 0;
  while (n % 2 == 0) {
    n /= 2;
    ++a;
  }
  // powers of two: prefer radix 8, then 4, avoid a lone 2 when possible
  int q = a / 3, r = a % 3;
  if (r == 1 && q >= 1) {
    --q;
    fac.push_back(4);
    fac.push_back(4);
  } else if (r == 1) {
    fac.push_back(2);
  } else if (r == 2) {
    fac.push_back(4);
  }
  for (int i = 0; i < q; ++i) fac.push_back(8);
  int b = 0;
  while (n % 3 == 0) {
    n /= 3;
    ++b;
  }
  for (int i = 0; i < b / 2; ++i) fac.push_back(9);
  if (b % 2) fac.push_back(3);
  for (int p : {5, 7, 11, 13}) {
    while (n % p == 0) {
      n /= p;
      fac.push_back(p);
    }
  }
  return n == 1;
}

static bool smooth7(int m) {
  for (int p : {2, 3, 5, 7})
    while (m % p == 0) m /= p;
  return m == 1;
}

// Bluestein length of the engine: the smallest M >= 2n - 1 of primes <= 7
static int bluestein_m(int n) {
  int M = 2 * n - 1;
  while (!smooth7(M)) ++M;
  return M;
}

static bool is_prime(int n) {
  if (n < 2) return false;
  for (int d = 2; d * d <= n; ++d)
    if (n % d == 0) return false;
  return true;
}

static long long powmod(long long b, long long e, long long m) {
  long long r = 1 % m;
  b %= m;
  while (e > 0) {
    if (e & 1) r = r * b % m;
    b = b * b % m;
    e >>= 1;
  }
  return r;
}

static int primitive_root(int n) {
  std::vector<int> pf;
  int m = n - 1;
  for (int d = 2; d * d <= m; ++d)
    if (m % d == 0) {
      pf.push_back(d);
      while (m % d == 0) m /= d;
    }
  if (m > 1) pf.push_back(m);
  for (int g = 2; g < n; ++g) {
    bool ok = true;
    for (int p : pf)
      if (powmod(g, (n - 1) / p, n) == 1) {
        ok = false;
        break;
      }
    if (ok) return g;
  }
  return -1;
}

static int tpl_for(int M, int n, const std::vector<int>& fac) {
  int need = (n + KEEP - 1) / KEEP;
  for (int R : fac) {
    const int nb = M / R;
    const int mb = std::max(1, kStage / R);
    need = std::max(need, (nb + mb - 1) / mb);
  }
  int t = 1;
  while (t < need) t <<= 1;
  return t;
}

static int dev_upload(void** dst, const void* src, size_t bytes, size_t* acc) {
  if (hipMalloc(dst, bytes) != hipSuccess) return fail(SPX_ERR_ALLOC, "hipMalloc of FFT tables");
  *acc += bytes;
  if (hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice) != hipSuccess)
    return fail(SPX_ERR_HIP, "hipMemcpy of FFT tables");
  return SPX_OK;
}

// upload a complex table in the plan's precision (csize 16: float64, 8: float32)
static int upload_table(void** dst, const std::vector<double>& v, int csize, size_t* acc) {
  if (csize == 16) return dev_upload(dst, v.data(), v.size() * sizeof(double), acc);
  std::vector<float> f(v.size());
  for (size_t i = 0; i < v.size(); ++i) f[i] = float(v[i]);
  return dev_upload(dst, f.data(), f.size() * sizeof(float), acc);
}

// naive long-double DFT of length M (used once per plan for the filters)
static void dft_ld(const std::vector<long double>& xr, const std::vector<long double>& xi,
                   const std::vector<long double>& wr, const std::vector<long double>& wi,
                   std::vector<double>& out, long double scale) {
  const int M = int(xr.size());
  out.assign(2 * size_t(M), 0.0);
  for (int k = 0; k < M; ++k) {
    long double sr = 0, si = 0;
    // idx = m k mod M, counted up: the 64-bit remainder took most of the time
    for (int m = 0, idx = 0; m < M; ++m, idx += idx + k < M ? k : k - M) {
      if (xr[m] == 0.0L && xi[m] == 0.0L) continue;
      sr += xr[m] * wr[idx] - xi[m] * wi[idx];
      si += xr[m] * wi[idx] + xi[m] * wr[idx];
    }
    out[2 * k] = double(sr * scale);
    out[2 * k + 1] = double(si * scale);
  }
}

// autotuner overrides (process-wide, read at plan creation)
static std::mutex g_tune_mu;
static std::map<std::pair<int, int>, LineTune> g_line_tune;
static std::map<int, WallTune> g_wall_tune;

void set_line_tune(int n, int csize, const LineTune& t) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_line_tune[{n, csize}] = t;
}
bool get_line_tune(int n, int csize, LineTune* t) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  auto it = g_line_tune.find({n, csize});
  if (it == g_line_tune.end()) return false;
  *t = it->second;
  return true;
}
void set_wall_tune(int n, const WallTune& t) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_wall_tune[n] = t;
}
bool get_wall_tune(int n, WallTune* t) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  auto it = g_wall_tune.find(n);
  if (it == g_wall_tune.end()) return false;
  *t = it->second;
  return true;
}
void clear_tunes() {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_line_tune.clear();
  g_wall_tune.clear();
}

int build_line_fft(LineFFTHost& f, int n, int csize, int want_lines, int max_block,
                   size_t lds_budget, int force_m) {
  std::vector<int> fac;
  f.n = n;
  if (force_m > 0) {
    f.mode = 1;
    f.M = force_m;
    factor_small(f.M, fac);
  } else if (factor_small(n, fac)) {
    f.mode = 0;
    f.M = n;
  } else if (is_prime(n) && factor_small(n - 1, fac)) {
    f.mode = 2;
    f.M = n - 1;
  } else {
    f.mode = 1;
    f.M = bluestein_m(n);
    factor_small(f.M, fac);
  }
  if (int(fac.size()) > kMaxStages) return fail(SPX_ERR_UNSUPPORTED, "FFT length has too many factors");
  f.nstage = int(fac.size());
  long long Ns = 1;
  for (int i = 0; i < f.nstage; ++i) {
    f.radix[i] = fac[i];
    f.magic[i] = Ns > 1 ? unsigned(((1ULL << 32) + Ns - 1) / Ns) : 0u;
    Ns *= fac[i];
  }
  // at least 2 threads per line: the wall kernels handle z = 0 and z = Lz on
  // lanes 0 and 1
  f.tpl = std::max(2, tpl_for(f.M, n, fac));
  LineTune tune;
  const bool tuned = get_line_tune(n, csize, &tune);
  auto pow2 = [](int v) { return v > 0 && (v & (v - 1)) == 0; };
  if (tuned && pow2(tune.threads) && tune.threads >= f.tpl && tune.threads <= kMaxBlock)
    f.tpl = tune.threads;
  if (f.tpl > kMaxBlock)
    return fail(SPX_ERR_UNSUPPORTED, "FFT length " + std::to_string(n) + " exceeds the LDS engine");
  f.lgtpl = 0;
  while ((1 << f.lgtpl) < f.tpl) ++f.lgtpl;
  const int span = f.mode == 0 ? n : (f.mode == 1 ? f.M : 2 * n);
  f.ldl = span + ((span % 16 == 0) ? 1 : 0);
  // tables staged in LDS: twiddles; Bluestein filter + chirp; Rader filter + indices
  if (f.mode == 0) f.tab = f.M;
  else if (f.mode == 1) f.tab = 2 * f.M + n;
  else f.tab = 2 * f.M + int((2 * size_t(f.M) * sizeof(int) + csize - 1) / csize);
  int nl = std::max(1, max_block / f.tpl);
  if (want_lines > 0) nl = std::min(nl, want_lines);
  while (nl > 1 && (size_t(f.tab) + size_t(nl) * f.ldl) * csize > lds_budget) nl >>= 1;
  // Rader / Bluestein: leave the filter / chirp / index tables in global
  // memory (L1/L2-resident) when staging them in LDS would cost workgroups
  // per CU, counted up to 4 per CU (beyond that registers bound the
  // occupancy of these kernels); kernels for this are built for radices <= 9
  bool small_radices = true;
  for (int R : fac) small_radices = small_radices && R <= 9;
  if (f.mode != 0 && small_radices) {
    const size_t lds_cu = 160 * 1024, lines = size_t(nl) * f.ldl;
    auto wgs = [&](size_t tab) {
      return std::min<size_t>(4, lds_cu / ((tab + lines) * size_t(csize)));
    };
    if (wgs(size_t(f.M)) > wgs(size_t(f.tab))) f.tab = f.M;
    if (tuned && tune.gtab == 1) f.tab = f.M;
    if (tuned && tune.gtab == 0 && f.tab == f.M)
      f.tab = f.mode == 1 ? 2 * f.M + n
                          : 2 * f.M + int((2 * size_t(f.M) * sizeof(int) + csize - 1) / csize);
  }
  if (tuned && pow2(tune.lines) && tune.lines * f.tpl <= kMaxBlock &&
      (size_t(f.tab) + size_t(tune.lines) * f.ldl) * csize <= 160 * 1024)
    nl = tune.lines;
  if ((size_t(f.tab) + size_t(nl) * f.ldl) * csize > 160 * 1024)
    return fail(SPX_ERR_UNSUPPORTED, "FFT line does not fit in LDS");
  f.nl = nl;
  f.lgnl = 0;
  while ((1 << f.lgnl) < f.nl) ++f.lgnl;
  // tables in long double
  const long double PI2 = 6.283185307179586476925286766559005768L;
  const int M = f.M;
  std::vector<long double> wr(M), wi(M);
  for (int m = 0; m < M; ++m) {
    wr[m] = cosl(PI2 * (long double)m / (long double)M);
    wi[m] = -sinl(PI2 * (long double)m / (long double)M);
  }
  std::vector<double> tw(2 * size_t(M));
  for (int m = 0; m < M; ++m) {
    tw[2 * m] = double(wr[m]);
    tw[2 * m + 1] = double(wi[m]);
  }
  int rc = upload_table(&f.tw, tw, csize, &f.bytes);
  if (rc) return rc;
  if (f.mode == 1) {
    // chirp w[m] = exp(-pi i (m^2 mod 2n)/n)
    const long double PI = PI2 / 2;
    std::vector<long double> cr(n), ci(n);
    std::vector<double> ch(2 * size_t(M), 0.0);  // zeros from n on (the wave plans read M entries)
    for (int m = 0; m < n; ++m) {
      const long long r = (long long)m * m % (2LL * n);
      cr[m] = cosl(PI * (long double)r / (long double)n);
      ci[m] = -sinl(PI * (long double)r / (long double)n);
      ch[2 * m] = double(cr[m]);
      ch[2 * m + 1] = double(ci[m]);
    }
    // b[m] = conj(w[|m|]) wrapped; bfil = DFT_M(b) / M
    std::vector<long double> br(M, 0.0L), bi(M, 0.0L);
    br[0] = cr[0];
    bi[0] = -ci[0];
    for (int m = 1; m < n; ++m) {
      br[m] = cr[m];
      bi[m] = -ci[m];
      br[M - m] = cr[m];
      bi[M - m] = -ci[m];
    }
    std::vector<double> bf;
    dft_ld(br, bi, wr, wi, bf, 1.0L / M);
    if ((rc = upload_table(&f.chirp, ch, csize, &f.bytes))) return rc;
    if ((rc = upload_table(&f.bfil, bf, csize, &f.bytes))) return rc;
  } else if (f.mode == 2) {
    // Rader: a_q = x[g^q], b_m = W_n^(g^-m), X[g^-p] = x0 + (a (*) b)_p
    const int g = primitive_root(n);
    if (g < 0) return fail(SPX_ERR_UNSUPPORTED, "no primitive root for Rader length");
    std::vector<int> perm(2 * size_t(M));
    const long long ginv = powmod(g, n - 2, n);
    for (int q = 0; q < M; ++q) {
      perm[q] = int(powmod(g, q, n));
      perm[M + q] = int(powmod(ginv, q, n));
    }
    std::vector<long double> br(M), bi(M);
    for (int m = 0; m < M; ++m) {
      const long double ang = PI2 * (long double)perm[M + m] / (long double)n;
      br[m] = cosl(ang);
      bi[m] = -sinl(ang);
    }
    std::vector<double> bf;
    dft_ld(br, bi, wr, wi, bf, 1.0L / M);
    if ((rc = upload_table(&f.bfil, bf, csize, &f.bytes))) return rc;
    if ((rc = dev_upload(&f.perm, perm.data(), perm.size() * sizeof(int), &f.bytes))) return rc;
  }
  return SPX_OK;
}

// sizes of the compiled plans, indexed by plan number
struct WaveInfo {
  int n, m, lanes, mode, nmax, ldl, tab, twm, lines16, lines8, npass;
  const int* radix;
  bool natural, xy;
  int lines(int csize) const { return csize == 16 ? lines16 : lines8; }
};
template <int W = 0>
static void wave_infos(WaveInfo* o) {
  using P = typename WavePlanN<W>::type;
  o[W] = WaveInfo{P::n,   P::m,   P::lanes,          P::mode,          P::nmax,  P::ldl,
                  P::tab, P::twm, wave_lines<W>(16), wave_lines<W>(8), P::npass, P::radix,
                  P::natural, P::xy};
  if constexpr (W + 1 < kWavePlans) wave_infos<W + 1>(o);
}
static const WaveInfo* wave_info() {
  static const struct Tab {
    WaveInfo t[kWavePlans];
    Tab() { wave_infos<>(t); }
  } tab;
  return tab.t;
}
// shape of a line plan run by compiled plan w, with the plan's table (the
// engine's W_M in the order of the passes, stage_twiddle, then W_9^0..4) in the
// place of the engine's
static int set_wave(LineFFTHost& h, int w, int csize) {
  const WaveInfo& i = wave_info()[w];
  h.wave = w;
  h.tpl = i.lanes;
  h.nl = i.lines(csize);
  for (h.lgtpl = 0; (1 << h.lgtpl) < h.tpl;) ++h.lgtpl;
  for (h.lgnl = 0; (1 << h.lgnl) < h.nl;) ++h.lgnl;
  h.ldl = i.ldl;
  h.tab = i.tab;  // staged in LDS; filter, chirp and indices in global memory
  // a tuned line count that fits beside what the kernels stage behind the lines:
  // float32 boundary planes (two times eight float64 values a line) and a sum per thread
  LineTune tune;
  if (get_line_tune(h.n, csize, &tune) && tune.lines > 0 && (tune.lines & (tune.lines - 1)) == 0 &&
      tune.lines * h.tpl >= 64 && tune.lines * h.tpl <= kMaxBlock) {
    const LineFFTHost t = h.with_lines(tune.lines);
    const size_t behind = csize == 8 ? size_t(t.nl) * 16 * 16 + 16 : size_t(t.nl) * t.tpl * 8;
    if (t.lds_bytes(size_t(csize)) + behind <= 160 * 1024) h = t;
  }
  if (i.natural) return SPX_OK;  // the engine's own table
  const long double PI2 = 6.283185307179586476925286766559005768L;
  const int M = h.M;
  std::vector<double> tw(2 * size_t(i.tab), 0.0);
  auto put = [&](int at, int m) {  // entry at <- W_M^m
    tw[2 * at] = double(cosl(PI2 * (long double)m / (long double)M));
    tw[2 * at + 1] = double(-sinl(PI2 * (long double)m / (long double)M));
  };
  int Ns = 1;
  for (int p = 0; p < i.npass; ++p) {
    const int R = i.radix[p];
    for (int r = 1; r < R; ++r)
      for (int jm = 0; jm < Ns; ++jm) put(r * Ns + jm - 1, r * jm * (M / (Ns * R)));
    Ns *= R;
  }
  if (M % 9 == 0)
    for (int q = 0; q < 5; ++q) put(M + q, q * (M / 9));
  if (h.tw) (void)hipFree(h.tw);
  h.tw = nullptr;
  h.bytes -= size_t(M) * csize;
  return upload_table(&h.tw, tw, csize, &h.bytes);
}

// The compiled plan of a z line: the direct or Rader plan of exactly this
// length; for the other lengths with a prime factor above 13 the smallest
// Bluestein M >= 2n - 1.  Rader lengths without a plan stay on the engine: its
// two (n-1)-point FFTs are more accurate in float32 (gradre's error at 89 and
// 281 1.53e-7 and 1.74e-7 through Bluestein, 1.26e-7 and 1.49e-7 through
// Rader), and smooth lengths without a plan because one FFT beats two.
// same_bits (mixed plans): only plans that run the engine's own arithmetic
// (its radices, table twiddles and Bluestein M), and those the lines always
// had.  The float32 nonlinear term's rounding is amplified by the pressure of
// the next stages, and a last-bit change anywhere redraws all of it (192^3,
// two steps: pressure 5e-6 in the norm, up to 1e-3 of its rms in single
// modes), so a mixed run keeps its bits instead.
int build_wave_fft(LineFFTHost& f, int n, int csize, bool same_bits) {
  f = LineFFTHost();
  if (const char* e = std::getenv("SPX_WAVE"))
    if (e[0] == '0') return SPX_OK;
  LineFFTHost h;
  std::vector<int> fac;
  const bool direct = factor_small(n, fac);
  const bool rader = !direct && is_prime(n) && factor_small(n - 1, fac);
  constexpr int kFixedZ = 3;  // plans 0 .. 2: z lines of 537, 539, 1049
  int w = -1;
  for (int q = 0; q < kWavePlans; ++q) {
    const WaveInfo& i = wave_info()[q];
    if (!i.lines(csize) || (same_bits && i.twm != 0 && i.n == 0)) continue;
    if (i.n == n && q < kFixedZ) {  // a plan of this length alone
      w = q;
      break;
    }
    if (i.n != 0) continue;
    if (direct) {
      if (i.mode == 0 && i.m == n) w = q;
    } else if (rader) {
      if (i.mode == 2 && i.m == n - 1) w = q;
    } else if (i.mode == 1 && n <= i.nmax && (w < 0 || i.m < wave_info()[w].m) &&
               (!same_bits || i.m == bluestein_m(n))) {
      w = q;
    }
  }
  if (w < 0) return SPX_OK;
  const int blu = wave_info()[w].mode == 1 ? wave_info()[w].m : 0;
  if (int rc = build_line_fft(h, n, csize, 0, 256, 64 * 1024, blu)) {
    free_line_fft(h);
    return rc;
  }
  if (int rc = set_wave(h, w, csize)) {
    free_line_fft(h);
    return rc;
  }
  f = h;
  return SPX_OK;
}

int attach_xy_wave(LineFFTHost& f, int csize) {
  for (const char* v : {"SPX_WAVE", "SPX_WAVE_XY"})
    if (const char* e = std::getenv(v))
      if (e[0] == '0') return SPX_OK;
  if (f.mode != 0) return SPX_OK;
  for (int q = 0; q < kWavePlans; ++q) {
    const WaveInfo& i = wave_info()[q];
    if (!i.xy || i.m != f.n || !i.lines(csize)) continue;
    if (!i.natural) return set_wave(f, q, csize);
    if (f.n == 512 && f.tpl == 64) f.wave = q;  // the engine's launch shape
    return SPX_OK;
  }
  return SPX_OK;
}

void free_line_fft(LineFFTHost& f) {
  if (f.tw) (void)hipFree(f.tw);
  if (f.chirp) (void)hipFree(f.chirp);
  if (f.bfil) (void)hipFree(f.bfil);
  if (f.perm) (void)hipFree(f.perm);
  f.tw = f.chirp = f.bfil = f.perm = nullptr;
  f.bytes = 0;
}
#endif  // SPX_PART 1 (plan tables)

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static inline dim3 blk(const LineFFTHost& f) { return dim3(unsigned(f.nl * f.tpl)); }

// Raise the dynamic-LDS limit of a kernel when a launch needs more than 64 KiB.
template <typename K>
static int lds_limit(K kernel, size_t bytes) {
  if (bytes <= 65536) return SPX_OK;
  SPX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes)));
  return SPX_OK;
}

// radix set of a plan: the smallest compiled kernel family that covers it
// (Rader and Bluestein plans never use the power-of-two family)
[[maybe_unused]] static int rset_of(const LineFFTHost& f) {
  if (f.wave >= 0) return RS_WAVE + f.wave;
  if (f.mode != 0 && f.tab == f.M) return RS_GTAB;  // radices <= 9 (build_line_fft)
  int rs = f.mode == 0 ? RS_POW2 : RS_SMOOTH;
  for (int i = 0; i < f.nstage; ++i) {
    const int R = f.radix[i];
    if (R == 11 || R == 13) rs = RS_ALL;
    else if (R != 2 && R != 4 && R != 8 && rs < RS_SMOOTH) rs = RS_SMOOTH;
  }
  return rs;
}

// fn(std::integral_constant<int, RS>) for the radix set of a general plan
template <typename F>
static int with_general(const LineFFTHost& f, F&& fn) {
  switch (rset_of(f)) {
    case RS_POW2: return fn(std::integral_constant<int, RS_POW2>{});
    case RS_SMOOTH: return fn(std::integral_constant<int, RS_SMOOTH>{});
    case RS_ALL: return fn(std::integral_constant<int, RS_ALL>{});
    case RS_GTAB: return fn(std::integral_constant<int, RS_GTAB>{});
    default: return fail(SPX_ERR_STATE, "wave line plan passed to a general kernel");
  }
}
// the same for any plan, compiled ones included, with csize-byte elements
template <int CS, bool XY, int W = 0, int END = kWavePlans, typename F>
static int with_wave(int w, F&& fn) {
  if constexpr (W < END) {
    if constexpr (wave_lines<W>(CS) > 0 && (!XY || WavePlanN<W>::type::xy)) {
      if (w == W) return fn(std::integral_constant<int, RS_WAVE + W>{});
    }
    return with_wave<CS, XY, W + 1, END>(w, fn);
  } else {
    return fail(SPX_ERR_STATE, "line plan without a compiled kernel family");
  }
}
template <int CS, typename F>
static int with_z(const LineFFTHost& f, F&& fn) {
  return f.wave >= 0 ? with_wave<CS, false>(f.wave, fn) : with_general(f, fn);
}
constexpr int kInplacePlans = 2;  // 1080 and 539
template <typename F>
[[maybe_unused]] static int with_inplace(const LineFFTHost& f, F&& fn) {
  return f.wave >= 0 ? with_wave<16, false, 0, kInplacePlans>(f.wave, fn) : with_general(f, fn);
}
// x / y lines: compiled plans of direct lengths
template <int CS, typename F>
static int with_xy(const LineFFTHost& f, F&& fn) {
  return f.wave >= 0 ? with_wave<CS, true>(f.wave, fn) : with_general(f, fn);
}
// f with fewer lines per workgroup where a launch of that many lines and
// fields would leave CUs idle: down to one wave, and to rows of 64 bytes where a
// workgroup's lines are neighbours in memory (least: lines of such a row).
// Two workgroups per CU: one step's kernels at limits of 0 / 256 / 512 / 1024 take
// 241 / 192 / 192 / 192 us for HD 32^3, 324 / 310 / 285 / 284 for 64^3, 572 / 565 / 559
// / 554 for 96x120x77, 95 / 90 / 84 / 86 for the 160x120x103 transforms.
// The engine's Rader and Bluestein lines keep theirs: a workgroup stages their filter
// and index tables too, which fewer threads do more slowly (x transforms of
// 54x50x71 10.3 -> 9.9 us back, 10.6 -> 10.4 forward, without this).
constexpr long kSpread = 512;
static inline LineFFTHost spread(const LineFFTHost& f, long lines, long fields, int least) {
  int nl = f.nl;
  if (f.wave < 0 && f.mode != 0) return f;
  while (nl > least && nl * f.tpl > 64 && (lines + nl - 1) / nl * fields < kSpread) nl >>= 1;
  return f.with_lines(nl);
}
#define SPX_COMMA ,
// launch the instance KER<TY, RS TARGS> of the dispatcher DISP(F, ...)
#define SPX_LAUNCH(DISP, F, KER, TY, TARGS, GRID, BLOCK, LDS, STREAM, ...)                   \
  do {                                                                                       \
    const int lrc_ = DISP(F, [&](auto rs_) -> int {                                          \
      constexpr int RS_ = decltype(rs_)::value;                                              \
      if (int rc_ = lds_limit(KER<TY SPX_COMMA RS_ TARGS>, (LDS))) return rc_;               \
      hipLaunchKernelGGL((KER<TY SPX_COMMA RS_ TARGS>), GRID, BLOCK, LDS, STREAM,            \
                         __VA_ARGS__);                                                       \
      return SPX_OK;                                                                         \
    });                                                                                      \
    if (lrc_) return lrc_;                                                                   \
  } while (0)
template <typename T>
static inline cpx<T>* C_(void* p) { return static_cast<cpx<T>*>(p); }
template <typename T>
static inline const cpx<T>* C_(const void* p) { return static_cast<const cpx<T>*>(p); }

// ---- transforms ----
// lo selects the float32 kernels and tables of a mixed plan.
// the z-transform plan: the wave variant where one is compiled
static inline const LineFFTHost& fzt(const spx_plan* p, bool lo) {
  if (lo) return p->fzw32.wave >= 0 ? p->fzw32 : p->fz32;
  return p->fzw.wave >= 0 ? p->fzw : p->fz;
}

[[maybe_unused]] static int check_lo(const spx_plan* p, bool lo) {
  if (lo && !p->fp32) return fail(SPX_ERR_STATE, "float32 kernels need a mixed-precision plan");
  return SPX_OK;
}

#if !defined(SPX_PART) || SPX_PART == 1
int zfft_inplace(spx_plan* p, void* S, int forward, int cont, double scale) {
  // the public one-dimensional transforms: compiled plans of the long lines only
  const LineFFTHost& f = p->fzw.wave >= 0 && p->fzw.wave < kInplacePlans ? p->fzw : p->fz;
  const long nlines = p->wlines();
  const unsigned nb = unsigned((nlines + f.nl - 1) / f.nl);
  const int C = p->g.Cz, d = p->g.oz;
  ProfScope ps_(p, "z_inplace", double(p->wnc()) * 2.0 * 16.0);
  SPX_LAUNCH(with_inplace, f, k_z_inplace, double, , dim3(nb), blk(f), f.lds_bytes(16), p->stream,
                C_<double>(S), nlines, f.dev<Cd>(), p->np, forward, (cont && C > 0) ? 1 : 0,
                scale, p->d_dir, C, d);
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}

int fc_continue_only(spx_plan* p, void* S) {
  const long nlines = p->wlines();
  const int C = p->g.Cz;
  if (C <= 0) return SPX_OK;
  const long tot = nlines * C;
  ProfScope ps_(p, "fc_continue", double(nlines) * 16.0 * (2 * p->g.oz + C));
  hipLaunchKernelGGL(k_fc_continue<double>, dim3(unsigned((tot + 255) / 256)), dim3(256), 0,
                     p->stream, C_<double>(S), nlines, p->g.nz, p->np, C, p->g.oz, p->d_dir);
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}

#endif  // SPX_PART 1 (z transforms in place)

template <typename T>
struct ZForward {
  static int run(spx_plan* p, int ncomp, const void* const* X, void* const* S, int nofft, const
                 LineFFTHost& f, const void* const* Xb);
};
template <typename T>
int ZForward<T>::run(spx_plan* p, int ncomp, const void* const* X, void* const* S, int nofft,
                      const LineFFTHost& fp, const void* const* Xb) {
  // members: grid.z; X holds np planes per member (all nz with nofft)
  const long pl = long(p->nkx) * p->g.ny;
  const LineFFTHost f = spread(fp, pl, long(ncomp) * p->mem, 64 / int(sizeof(cpx<T>)));
  dim3 grid(unsigned((pl + f.nl - 1) / f.nl), unsigned(ncomp), unsigned(p->mem));
  const long xstride = pl * (nofft ? p->g.nz : p->np);
  ZX2S<T> a;
  for (int c = 0; c < kMaxComp; ++c) {
    a.x[c] = c < ncomp ? C_<T>(X[c]) : nullptr;
    a.s[c] = c < ncomp ? C_<T>(S[c]) : nullptr;
    a.xb[c] = c < ncomp && Xb ? C_<double>(Xb[c]) : nullptr;
  }
  ProfScope ps_(p, "z_x2s", double(p->wkx()) * p->g.ny * sizeof(cpx<T>) * ncomp *
                                ((nofft ? p->g.nz : p->np) + p->g.nz));
  if constexpr (sizeof(T) == 4) if (Xb) {
    // plus the staged float64 boundary values of the tile (nl * 2d, aligned)
    const size_t bnd_stage_bytes = size_t(f.nl) * 2 * p->g.oz * sizeof(Cd) + 16;
    SPX_LAUNCH(with_z<sizeof(cpx<T>)>, f, k_z_x2s, T, SPX_COMMA true, grid, blk(f),
                  f.lds_bytes(sizeof(cpx<T>)) + bnd_stage_bytes, p->stream, a,
                  f.dev<cpx<T>>(), p->nkx, p->g.ny, p->np, nofft, p->d_dir, p->g.Cz, p->g.oz,
                  xstride);
    SPX_CHECK_LAUNCH();
    return SPX_OK;
  }
  SPX_LAUNCH(with_z<sizeof(cpx<T>)>, f, k_z_x2s, T, SPX_COMMA false, grid, blk(f), f.lds_bytes(sizeof(cpx<T>)),
                p->stream, a, f.dev<cpx<T>>(), p->nkx, p->g.ny, p->np, nofft, p->d_dir,
                p->g.Cz, p->g.oz, xstride);
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}
#if !defined(SPX_PART) || SPX_PART == 4
template struct ZForward<double>;
#else
extern template struct ZForward<double>;
#endif
#if !defined(SPX_PART) || SPX_PART == 5
template struct ZForward<float>;
#else
extern template struct ZForward<float>;
#endif
#if !defined(SPX_PART) || SPX_PART == 1
int zfft_x2s(spx_plan* p, int ncomp, const void* const* X, void* const* S, int nofft, bool lo,
             const void* const* Xb) {
  if (int rc = check_lo(p, lo)) return rc;
  if (ncomp < 1 || ncomp > kMaxComp) return fail(SPX_ERR_ARG, "zfft_x2s: bad field count");
  if (Xb && (nofft || p->g.Cz <= 0)) return fail(SPX_ERR_ARG, "boundary planes need a continuation");
  if (!lo && Xb) return fail(SPX_ERR_ARG, "boundary planes: float32 transforms only");
  return lo ? ZForward<float>::run(p, ncomp, X, S, nofft, fzt(p, true), Xb)
            : ZForward<double>::run(p, ncomp, X, S, nofft, fzt(p, false), Xb);
}

int zfft_s2x_bnd(spx_plan* p, const void* const* S, int ncomp, void* XVb, void* XZb) {
  if (!p->d_wbnd) return fail(SPX_ERR_STATE, "plan has no boundary-plane table");
  if (ncomp < 1 || ncomp > 4) return fail(SPX_ERR_ARG, "zfft_s2x_bnd: 1..4 components");
  BndSrc src;
  for (int c = 0; c < 4; ++c) src.s[c] = c < ncomp ? C_<double>(S[c]) : nullptr;
  const long lines = p->wlines();
  const dim3 grid(unsigned((lines + 15) / 16), unsigned(ncomp));
  ProfScope ps_(p, "z_s2x", double(ncomp) * double(p->wnc()) * 16.0);
  const int n = p->g.nz, nkx = p->nkx, ny = p->g.ny, mem = p->mem;
  const Cd* w1 = static_cast<const Cd*>(p->d_wbnd);
  const Cd* wt = w1 + n;
  Cd* v = C_<double>(XVb);
  Cd* z = C_<double>(XZb);
  switch (p->g.oz) {
#define SPX_BND_CASE(D)                                                                        \
  case D:                                                                                      \
    hipLaunchKernelGGL((k_z_s2x_bnd<D, 2>), grid, dim3(256), 0, p->stream, src, v, z, w1, wt, n, \
                       nkx, ny, mem, p->d_kz);                                                 \
    break;
    SPX_BND_CASE(1)
    SPX_BND_CASE(2)
    SPX_BND_CASE(3)
    SPX_BND_CASE(4)
    SPX_BND_CASE(5)
    SPX_BND_CASE(6)
    SPX_BND_CASE(7)
    SPX_BND_CASE(8)
#undef SPX_BND_CASE
    default:
      return fail(SPX_ERR_UNSUPPORTED, "boundary planes: matching order above 8");
  }
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}

#endif  // SPX_PART 1

// S is float64 in both precisions; X (and X2) are T
template <typename T>
struct ZBackward {
  static int run(spx_plan* p, int ncomp, const void* const* S, void* const* X, int dirn, int
                 nzout, int nofft, void* const* X2, const LineFFTHost& f);
};
template <typename T>
int ZBackward<T>::run(spx_plan* p, int ncomp, const void* const* S, void* const* X, int dirn,
                      int nzout, int nofft, void* const* X2, const LineFFTHost& fp) {
  // members: grid.z; X holds nzout planes per member
  const long pl = long(p->nkx) * p->g.ny;
  const LineFFTHost f = spread(fp, pl, long(ncomp) * p->mem, 64 / int(sizeof(cpx<T>)));
  dim3 grid(unsigned((pl + f.nl - 1) / f.nl), unsigned(ncomp), unsigned(p->mem));
  const double line = double(p->wkx()) * p->g.ny * ncomp;
  ZS2X<T, double> a;
  for (int c = 0; c < kMaxComp; ++c) {
    a.s[c] = c < ncomp ? C_<double>(S[c]) : nullptr;
    a.x[c] = c < ncomp ? C_<T>(X[c]) : nullptr;
    a.x2[c] = c < ncomp && X2 ? C_<T>(X2[c]) : nullptr;
  }
  if (X2) {
    ProfScope ps_(p, "z_s2x_dual", line * (16.0 * p->g.nz + 2.0 * sizeof(cpx<T>) * nzout));
    SPX_LAUNCH(with_z<sizeof(cpx<T>)>, f, k_z_s2x, T, SPX_COMMA true SPX_COMMA double, grid, blk(f),
                  f.lds_bytes(sizeof(cpx<T>)), p->stream, a, f.dev<cpx<T>>(), p->nkx, p->g.ny,
                  nzout, dirn, nofft, p->d_kx, p->d_ky, p->d_kz);
  } else {
    ProfScope ps_(p, "z_s2x", line * (16.0 * p->g.nz + sizeof(cpx<T>) * nzout));
    SPX_LAUNCH(with_z<sizeof(cpx<T>)>, f, k_z_s2x, T, SPX_COMMA false SPX_COMMA double, grid, blk(f),
                  f.lds_bytes(sizeof(cpx<T>)), p->stream, a, f.dev<cpx<T>>(), p->nkx, p->g.ny,
                  nzout, dirn, nofft, p->d_kx, p->d_ky, p->d_kz);
  }
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}
#if !defined(SPX_PART) || SPX_PART == 6
template struct ZBackward<double>;
#else
extern template struct ZBackward<double>;
#endif
#if !defined(SPX_PART) || SPX_PART == 7
template struct ZBackward<float>;
#else
extern template struct ZBackward<float>;
#endif
#if !defined(SPX_PART) || SPX_PART == 1
int zfft_s2x(spx_plan* p, int ncomp, const void* const* S, void* const* X, int dirn, int nzout,
             int nofft, void* const* X2, bool lo) {
  if (int rc = check_lo(p, lo)) return rc;
  if (ncomp < 1 || ncomp > kMaxComp) return fail(SPX_ERR_ARG, "zfft_s2x: bad field count");
  return lo ? ZBackward<float>::run(p, ncomp, S, X, dirn, nzout, nofft, X2, fzt(p, true))
            : ZBackward<double>::run(p, ncomp, S, X, dirn, nzout, nofft, X2, fzt(p, false));
}
#endif  // SPX_PART 1 (z transforms)

template <typename T>
struct YPass {
  static int run(spx_plan* p, int nf, const void* const* in, void* const* out, int forward, int
                 nplanes, void* const* Y2, const LineFFTHost& f, bool cont);
};
template <typename T>
int YPass<T>::run(spx_plan* p, int nf, const void* const* in, void* const* out, int forward,
                  int nplanes, void* const* Y2, const LineFFTHost& fp, bool cont) {
  // members are consecutive blocks of nplanes planes
  const long nlines = long(p->nkx) * nplanes * p->mem;
  const LineFFTHost f = spread(fp, nlines, nf, 64 / int(sizeof(cpx<T>)));
  dim3 grid(unsigned((nlines + f.nl - 1) / f.nl), unsigned(nf));
  YFields<T> a;
  int nd = 0;
  for (int c = 0; c < kMaxComp; ++c) {
    a.in[c] = c < nf ? C_<T>(in[c]) : nullptr;
    a.out[c] = c < nf ? C_<T>(out[c]) : nullptr;
    a.y2[c] = c < nf && Y2 ? C_<T>(Y2[c]) : nullptr;
    nd += a.y2[c] != nullptr;
  }
  const double io = double(nlines) * p->g.ny * sizeof(cpx<T>);
  if (nd > 0) {
    if (forward) return fail(SPX_ERR_ARG, "dual y transform is backward only");
    ProfScope ps_(p, "y_dual", io * (2.0 * nf + nd));
    SPX_LAUNCH(with_xy<sizeof(cpx<T>)>, f, k_y, T, SPX_COMMA true, grid, blk(f), f.lds_bytes(sizeof(cpx<T>)),
                  p->stream, a, f.dev<cpx<T>>(), p->nkx, p->g.ny, nlines, forward, p->d_ky,
                  p->npy, 0, 0, static_cast<const double*>(nullptr));
  } else {
    ProfScope ps_(p, "y", io * 2.0 * nf);
    SPX_LAUNCH(with_xy<sizeof(cpx<T>)>, f, k_y, T, SPX_COMMA false, grid, blk(f), f.lds_bytes(sizeof(cpx<T>)),
                  p->stream, a, f.dev<cpx<T>>(), p->nkx, p->g.ny, nlines, forward, p->d_ky,
                  p->npy, cont ? p->Cy : 0, p->oy, p->d_diry);
  }
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}
#if !defined(SPX_PART) || SPX_PART == 2
template struct YPass<double>;
#else
extern template struct YPass<double>;
#endif
#if !defined(SPX_PART) || SPX_PART == 9
template struct YPass<float>;
#else
extern template struct YPass<float>;
#endif
#if !defined(SPX_PART) || SPX_PART == 1
int yfft(spx_plan* p, int nf, const void* const* in, void* const* out, int forward, int nplanes,
         void* const* Y2, bool lo, bool cont) {
  if (int rc = check_lo(p, lo)) return rc;
  if (nf < 1 || nf > kMaxComp) return fail(SPX_ERR_ARG, "yfft: bad field count");
  if (cont && (!forward || p->Cy <= 0 || Y2))
    return fail(SPX_ERR_ARG, "y continuation: forward transforms of plans with Cy > 0 only");
  return lo ? YPass<float>::run(p, nf, in, out, forward, nplanes, Y2, p->fy32, cont)
            : YPass<double>::run(p, nf, in, out, forward, nplanes, Y2, p->fy, cont);
}

#endif  // SPX_PART 1

template <typename T>
static XFields<T> x_fields(int nf, const void* const* in, void* const* out) {
  XFields<T> a;
  for (int c = 0; c < kMaxComp; ++c) {
    a.in[c] = c < nf ? in[c] : nullptr;
    a.out[c] = c < nf ? out[c] : nullptr;
  }
  return a;
}

#if !defined(SPX_PART) || SPX_PART == 10
int xr2c(spx_plan* p, int nf, const void* const* R, void* const* X, int nplanes) {
  if (nf < 1 || nf > kMaxComp) return fail(SPX_ERR_ARG, "xr2c: bad field count");
  const long npairs = long(p->g.ny) * nplanes * p->mem / 2;
  const LineFFTHost f = spread(p->fx, npairs, nf, 1);
  const XFields<double> a = x_fields<double>(nf, R, X);
  ProfScope ps_(p, "xr2c", double(p->g.ny) * nplanes * p->mem * nf *
                               (8.0 * p->g.nx + 16.0 * p->nkx));
  const int rc = with_xy<16>(f, [&](auto rs) -> int {
    constexpr int RS = decltype(rs)::value;
    const size_t lds = f.lds_bytes(16);
    if (int lrc = lds_limit(k_xr2c<RS>, lds)) return lrc;
    hipLaunchKernelGGL(k_xr2c<RS>, dim3(unsigned((npairs + f.nl - 1) / f.nl), unsigned(nf)),
                       blk(f), lds, p->stream, a, f.dev<Cd>(), p->nkx, npairs);
    return SPX_OK;
  });
  if (rc) return rc;
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}
#endif

template <typename T>
struct XBackward {
  static int run(spx_plan* p, int nf, const void* const* X, void* const* R, int nplanes, int
                 dirx, const LineFFTHost& f);
};
template <typename T>
int XBackward<T>::run(spx_plan* p, int nf, const void* const* X, void* const* R, int nplanes,
                  int dirx, const LineFFTHost& fp) {
  const long npairs = long(p->g.ny) * nplanes * p->mem / 2;
  const LineFFTHost f = spread(fp, npairs, nf, 1);
  dim3 grid(unsigned((npairs + f.nl - 1) / f.nl), unsigned(nf));
  const XFields<T> a = x_fields<T>(nf, X, R);
  ProfScope ps_(p, "xc2r", double(p->g.ny) * nplanes * p->mem * nf *
                               (double(sizeof(T)) * p->g.nx + double(sizeof(cpx<T>)) * p->nkx));
  SPX_LAUNCH(with_xy<sizeof(cpx<T>)>, f, k_xc2r, T, , grid, blk(f), f.lds_bytes(sizeof(cpx<T>)), p->stream, a,
                f.dev<cpx<T>>(), p->nkx, npairs, dirx, p->d_kx);
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}
#if !defined(SPX_PART) || SPX_PART == 10
template struct XBackward<double>;
#else
extern template struct XBackward<double>;
#endif
#if !defined(SPX_PART) || SPX_PART == 11
template struct XBackward<float>;
#else
extern template struct XBackward<float>;
#endif
#if !defined(SPX_PART) || SPX_PART == 1
int xc2r(spx_plan* p, int nf, const void* const* X, void* const* R, int nplanes, int dirx,
         bool lo) {
  if (int rc = check_lo(p, lo)) return rc;
  if (nf < 1 || nf > kMaxComp) return fail(SPX_ERR_ARG, "xc2r: bad field count");
  return lo ? XBackward<float>::run(p, nf, X, R, nplanes, dirx, p->fx32)
            : XBackward<double>::run(p, nf, X, R, nplanes, dirx, p->fx);
}
#endif

#if !defined(SPX_PART) || SPX_PART == 10
int xround(spx_plan* p, void* X) {
  const long npairs = long(p->g.ny) * p->np * p->mem / 2;
  const LineFFTHost f = spread(p->fx, npairs, 1, 1);
  ProfScope ps_(p, "xround", 4.0 * npairs * sizeof(Cd) * p->nkx);
  const int rc = with_xy<16>(f, [&](auto rs) -> int {
    constexpr int RS = decltype(rs)::value;
    const size_t lds = f.lds_bytes(16);
    if (int lrc = lds_limit(k_xround<RS>, lds)) return lrc;
    hipLaunchKernelGGL(k_xround<RS>, dim3(unsigned((npairs + f.nl - 1) / f.nl)), blk(f), lds,
                       p->stream, C_<double>(X), f.dev<Cd>(), p->nkx, npairs, double(p->g.ny),
                       double(p->g.nz));
    return SPX_OK;
  });
  if (rc) return rc;
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}

bool xcross_fused(const spx_plan* p) {
  if (p->fp32 || !p->XV[0] || p->fx.wave < 0) return false;
  return with_xy<16>(p->fx, [](auto rs) -> int { return xcross_ok<decltype(rs)::value>(); }) == 1;
}

int xcross(spx_plan* p, void* const* A, void* const* B, void* const* out) {
  const long npairs = long(p->g.ny) * p->np * p->mem / 2;
  const LineFFTHost f = spread(p->fx, npairs, 1, 1);
  const double tmp = 1.0 / std::pow(double(p->g.nx) * double(p->g.ny) * double(p->g.nz), 2);
  XCross a;
  for (int c = 0; c < 3; ++c) {
    a.a[c] = C_<double>(static_cast<const void*>(A[c]));
    a.b[c] = C_<double>(static_cast<const void*>(B[c]));
    a.out[c] = C_<double>(out[c]);
  }
  ProfScope ps_(p, "xcross", 18.0 * npairs * sizeof(Cd) * p->nkx);
  const int rc = with_xy<16>(f, [&](auto rs) -> int {
    constexpr int RS = decltype(rs)::value;
    if constexpr (xcross_ok<RS>()) {
      const size_t lds = f.lds_bytes(16);
      if (int lrc = lds_limit(k_xcross<RS>, lds)) return lrc;
      hipLaunchKernelGGL(k_xcross<RS>, dim3(unsigned((npairs + f.nl - 1) / f.nl)), blk(f), lds,
                         p->stream, a, f.dev<Cd>(), p->nkx, npairs, tmp);
      return SPX_OK;
    } else {
      return SPX_ERR_UNSUPPORTED;
    }
  });
  if (rc) return rc;
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}
#endif

template <typename T>
struct XGradProd {
  static int run(spx_plan* p, int nf, const void* const* YV, const void* const* YY, const void*
                 const* XZ, const void* const* vel, void* const* out, const LineFFTHost& f, int
                 nplanes);
};
template <typename T>
int XGradProd<T>::run(spx_plan* p, int nf, const void* const* YV, const void* const* YY,
                        const void* const* XZ, const void* const* vel, void* const* out,
                        const LineFFTHost& fp, int nplanes) {
  const long npairs = long(p->g.ny) * nplanes * p->mem / 2;
  const LineFFTHost f = spread(fp, npairs, nf, 1);
  dim3 grid(unsigned((npairs + f.nl - 1) / f.nl), unsigned(nf));
  const double t = double(p->g.nx) * double(p->g.ny) * double(p->g.nz);
  const double rows = double(p->g.ny) * nplanes * p->mem * nf;
  XProd<T> a;
  for (int c = 0; c < 4; ++c) {
    a.yv[c] = c < nf ? C_<T>(YV[c]) : nullptr;
    a.yy[c] = c < nf ? C_<T>(YY[c]) : nullptr;
    a.xz[c] = c < nf ? C_<T>(XZ[c]) : nullptr;
    a.out[c] = c < nf ? C_<T>(out[c]) : nullptr;
  }
  for (int c = 0; c < 3; ++c) a.vel[c] = static_cast<const T*>(vel[c]);
  ProfScope ps_(p, "xgrad_prod", rows * (4.0 * sizeof(cpx<T>) * p->nkx +
                                         3.0 * sizeof(T) * p->g.nx));
  SPX_LAUNCH(with_xy<sizeof(cpx<T>)>, f, k_xgrad_prod, T, , grid, blk(f), f.lds_bytes(sizeof(cpx<T>)), p->stream, a,
                f.dev<cpx<T>>(), p->nkx, npairs, 1.0 / (t * t), p->d_kx);
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}
#if !defined(SPX_PART) || SPX_PART == 12
template struct XGradProd<double>;
#else
extern template struct XGradProd<double>;
#endif
#if !defined(SPX_PART) || SPX_PART == 13
template struct XGradProd<float>;
#else
extern template struct XGradProd<float>;
#endif
template <typename T>
struct XGradFused {
  static int run(spx_plan* p, int nf, void* const* YV, void* const* YY, void* const* XZ,
                 void* const* out, const LineFFTHost& f);
};
template <typename T>
int XGradFused<T>::run(spx_plan* p, int nf, void* const* YV, void* const* YY, void* const* XZ,
                         void* const* out, const LineFFTHost& fp) {
  const int nplanes = p->np;
  const long npairs = long(p->g.ny) * nplanes * p->mem / 2;
  const LineFFTHost f = spread(fp, npairs, 1, 1);
  const double t = double(p->g.nx) * double(p->g.ny) * double(p->g.nz);
  const double rows = double(p->g.ny) * nplanes * p->mem;
  XGradArgs<T> a;
  for (int c = 0; c < 4; ++c) {
    a.yv[c] = c < nf ? C_<T>(static_cast<const void*>(YV[c])) : nullptr;
    a.yy[c] = c < nf ? C_<T>(static_cast<const void*>(YY[c])) : nullptr;
    a.xz[c] = c < nf ? C_<T>(static_cast<const void*>(XZ[c])) : nullptr;
    a.out[c] = c < nf ? C_<T>(out[c]) : nullptr;
  }
  ProfScope ps_(p, "xgrad_fused", rows * 4.0 * nf * sizeof(cpx<T>) * p->nkx);
  const int rc = with_xy<sizeof(cpx<T>)>(f, [&](auto rs) -> int {
    constexpr int RS = decltype(rs)::value;
    if constexpr (xfused_ok<RS>()) {
      const size_t lds = f.lds_bytes(sizeof(cpx<T>));
      if (int lrc = lds_limit(k_xgrad_fused<T, RS>, lds)) return lrc;
      const unsigned tiles = unsigned((npairs + f.nl - 1) / f.nl);
      hipLaunchKernelGGL((k_xgrad_fused<T, RS>), dim3(tiles, tiles < kSpread ? nf : 1), blk(f),
                         lds, p->stream, a, f.dev<cpx<T>>(), p->nkx, npairs, nf, 1.0 / (t * t),
                         p->d_kx);
      return SPX_OK;
    } else {
      return SPX_ERR_UNSUPPORTED;
    }
  });
  if (rc) return rc;
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}
#if !defined(SPX_PART) || SPX_PART == 14
template struct XGradFused<double>;
#else
extern template struct XGradFused<double>;
#endif
#if !defined(SPX_PART) || SPX_PART == 15
template struct XGradFused<float>;
#else
extern template struct XGradFused<float>;
#endif
#if !defined(SPX_PART) || SPX_PART == 1
int xgrad_fused(spx_plan* p, int nf, void* const* YV, void* const* YY, void* const* XZ,
                void* const* out, bool lo) {
  if (int rc = check_lo(p, lo)) return rc;
  if (nf < 3 || nf > 4) return fail(SPX_ERR_ARG, "xgrad_fused: 3 or 4 fields");
  return lo ? XGradFused<float>::run(p, nf, YV, YY, XZ, out, p->fx32)
            : XGradFused<double>::run(p, nf, YV, YY, XZ, out, p->fx);
}
#endif

#if !defined(SPX_PART) || SPX_PART == 1
int xgrad_prod(spx_plan* p, int nf, const void* const* YV, const void* const* YY,
               const void* const* XZ, const void* const* vel, void* const* out, bool lo,
               int nplanes) {
  if (int rc = check_lo(p, lo)) return rc;
  if (nf < 1 || nf > 4) return fail(SPX_ERR_ARG, "xgrad_prod: 1..4 fields");
  if (nplanes < 0) nplanes = p->np;
  return lo ? XGradProd<float>::run(p, nf, YV, YY, XZ, vel, out, p->fx32, nplanes)
            : XGradProd<double>::run(p, nf, YV, YY, XZ, vel, out, p->fx, nplanes);
}
#endif

#if !defined(SPX_PART) || SPX_PART == 3
// ---- float64 boundary / projection / diagnostics kernels ----
static int noslip_launch(spx_plan* p, void* vx, void* vy, const void* pr, const WallParams& wp,
                         int ncomp, const char* name, const RkLoad* rk) {
  if (p->wall.on) return wall_mfma(p, vx, vy, pr, wp, ncomp, rk);
  const LineFFTHost& f = p->fz;
  const long nlines = p->wlines();
  dim3 grid(unsigned((nlines + f.nl - 1) / f.nl), unsigned(ncomp));
  RkLoad r;
  std::memset(&r, 0, sizeof(r));
  if (rk) r = *rk;
  const double extra = rk ? (rk->nl32 ? 8.0 : 16.0) + 32.0 : 0.0;  // nl, c0, f reads
  ProfScope ps_(p, rk ? "noslip_rk" : name,
                ncomp * double(p->wnc()) * (2.0 * 16.0 + extra));
  SPX_LAUNCH(with_general, f, k_noslip, double, , grid, blk(f), f.lds_bytes(16), p->stream, C_<double>(vx),
                C_<double>(vy), C_<double>(pr), f.dev<Cd>(), nlines, p->g.ny, p->np,
                1.0 / double(p->g.nz), wp, p->d_kx, p->d_ky, p->d_dir, p->g.Cz, p->g.oz, r,
                rk ? 1 : 0);
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}

int noslip_fused(spx_plan* p, void* vx, void* vy, const void* pr, double tau,
                 const double vzsta[2], const double vzend[2], const RkLoad* rk) {
  WallParams wp;
  wp.tau = tau;
  wp.vb[0][0] = vzsta ? vzsta[0] : 0.0;
  wp.vb[1][0] = vzsta ? vzsta[1] : 0.0;
  wp.vb[0][1] = vzend ? vzend[0] : 0.0;
  wp.vb[1][1] = vzend ? vzend[1] : 0.0;
  wp.nxny = double(p->g.nx * p->g.ny);
  wp.scalar = 0;
  return noslip_launch(p, vx, vy, pr, wp, 2, "noslip", rk);
}


int sconst_fused(spx_plan* p, void* th) {
  WallParams wp;
  std::memset(&wp, 0, sizeof(wp));
  wp.scalar = 1;
  return noslip_launch(p, th, th, nullptr, wp, 1, "sconst", nullptr);
}


int pressure_walls(spx_plan* p, void* d) {
  const long nlines = p->wlines();
  ProfScope ps_(p, "pressure_walls", double(nlines) * 6.0 * 16.0);
  hipLaunchKernelGGL(k_pressure_walls, dim3(unsigned((nlines + 255) / 256)), dim3(256), 0,
                     p->stream, C_<double>(d), C_<double>(p->bc), C_<double>(p->pw), nlines,
                     p->g.nz, p->np, p->g.Lz, p->d_khom, p->d_z);
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}

// The two harmonic profiles of each distinct khom value, continued and
// transformed on the host in long double and rounded once to float64: rows
// 2u, 2u+1 of tab.  The table is reused by every line with that kh, every
// stage and every step, so its rounding acts as a systematic error of the
// projection; a float64 device FFT leaves several ulps in each entry and
// moves cfg1 (64^3, 100 steps) 4x further from the exact trajectory than
// per-line transforms do, a correctly rounded table does not.  Real input:
// P[nz-k] = conj(P[k]).  Threads over the profiles.
static void harmonic_table_ld(const std::vector<double>& khv, int n, int np, int C, int d,
                              const std::vector<double>& z, double Lz,
                              const std::vector<double>& dir, std::vector<double>& out) {
  const long double PI2 = 6.283185307179586476925286766559005768L;
  std::vector<long double> wr(n), wi(n);
  for (int m = 0; m < n; ++m) {
    wr[m] = cosl(PI2 * (long double)m / (long double)n);
    wi[m] = -sinl(PI2 * (long double)m / (long double)n);
  }
  const int U = int(khv.size());
  out.assign(size_t(2) * U * n * 2, 0.0);
  auto work = [&](int u0, int u1) {
    std::vector<long double> x(n);
    for (int u = u0; u < u1; ++u) {
      const long double kh = khv[u];
      for (int which = 0; which < 2; ++which) {
        for (int k = 0; k < np; ++k) {
          const long double zk = z[k];
          if (kh == 0.0L) x[k] = which == 0 ? zk : 1.0L;
          else x[k] = which == 0 ? expl(kh * (zk - (long double)Lz)) : expl(-kh * zk);
        }
        // FC-Gram continuation (fftp.fpp:755-773 order)
        const int top = np - d;
        for (int ii = 0; ii < C; ++ii) {
          const double* D0 = dir.data() + size_t(ii) * d;
          const double* D1 = dir.data() + size_t(C - 1 - ii) * d;
          long double a = (long double)D0[0] * x[top] + (long double)D1[0] * x[d - 1];
          for (int jj = 1; jj < d; ++jj) {
            a += (long double)D0[jj] * x[top + jj];
            a += (long double)D1[jj] * x[d - 1 - jj];
          }
          x[np + ii] = a;
        }
        double* o = out.data() + (size_t(2) * u + which) * n * 2;
        for (int k = 0; k <= n / 2; ++k) {
          long double sr = 0, si = 0;
          int idx = 0;
          for (int m = 0; m < n; ++m) {
            sr += x[m] * wr[idx];
            si += x[m] * wi[idx];
            idx += k;
            if (idx >= n) idx -= n;
          }
          o[2 * k] = double(sr);
          o[2 * k + 1] = double(si);
          if (k > 0 && n - k != k) {
            o[2 * (n - k)] = double(sr);
            o[2 * (n - k) + 1] = double(-si);
          }
        }
      }
    }
  };
  const int nt = std::max(1, std::min(16, int(std::thread::hardware_concurrency())));
  std::vector<std::thread> th;
  const int chunk = (U + nt - 1) / nt;
  for (int t = 0; t < nt; ++t) {
    const int u0 = t * chunk, u1 = std::min(U, u0 + chunk);
    if (u0 < u1) th.emplace_back(work, u0, u1);
  }
  for (auto& t : th) t.join();
}

int build_harmonic_table(spx_plan* p) {
  // SPX_HARMONIC_TABLE=0: no table (the harmonic kernel transforms per line;
  // for plans whose memory is tighter than 2 * (distinct kh) * nz complex values)
  if (const char* e = std::getenv("SPX_HARMONIC_TABLE"))
    if (e[0] == '0') return SPX_OK;
  const int n = p->g.nz, np = p->np, ny = p->g.ny;
  const size_t lines1 = size_t(p->nkx) * ny;
  std::unordered_map<uint64_t, int> seen;
  std::vector<double> khv;
  std::vector<int> idx(lines1 * size_t(p->nb));
  for (size_t l = 0; l < lines1; ++l) {
    uint64_t key;
    std::memcpy(&key, &p->h_khom[l], sizeof(key));
    auto it = seen.find(key);
    if (it == seen.end()) {
      it = seen.emplace(key, int(khv.size())).first;
      khv.push_back(p->h_khom[l]);
    }
    idx[l] = it->second;
  }
  for (int b = 1; b < p->nb; ++b)
    std::copy(idx.begin(), idx.begin() + long(lines1), idx.begin() + long(b * lines1));
  const int U = int(khv.size());
  void *tab = nullptr, *hid = nullptr, *kv = nullptr;
  const size_t tab_bytes = 2 * size_t(U) * n * sizeof(Cd);
  if (hipMalloc(&tab, tab_bytes) != hipSuccess) {
    (void)hipGetLastError();  // no table: proj_harmonic transforms per line
    return SPX_OK;
  }
  p->owned.push_back(tab);
  p->dev_bytes += tab_bytes;
  SPX_HIP(hipMalloc(&hid, idx.size() * sizeof(int)));
  p->owned.push_back(hid);
  p->dev_bytes += idx.size() * sizeof(int);
  SPX_HIP(hipMalloc(&kv, khv.size() * sizeof(double)));
  SPX_HIP(hipMemcpy(hid, idx.data(), idx.size() * sizeof(int), hipMemcpyHostToDevice));
  SPX_HIP(hipMemcpy(kv, khv.data(), khv.size() * sizeof(double), hipMemcpyHostToDevice));
  // long double on the host (the default; about 2 U np nz / 2 multiply-adds,
  // split over up to 16 threads), or the profiles continued and transformed
  // on the device in float64 for tables whose host cost would be too high
  // (U nz^2 > 2e11, e.g. 1024^3) or with SPX_HARMONIC_LD=0
  bool host_ld = double(U) * double(n) * double(n) <= 2e11;
  if (const char* e = std::getenv("SPX_HARMONIC_LD")) host_ld = e[0] != '0';
  if (host_ld) {
    std::vector<double> h;
    harmonic_table_ld(khv, n, np, p->g.Cz, p->g.oz, p->h_z, p->g.Lz, p->h_dir, h);
    SPX_HIP(hipMemcpy(tab, h.data(), tab_bytes, hipMemcpyHostToDevice));
  } else {
    const long tot = long(U) * np;
    hipLaunchKernelGGL(k_harm_profiles, dim3(unsigned((tot + 255) / 256)), dim3(256), 0,
                       p->stream, static_cast<Cd*>(tab), static_cast<const double*>(kv), U, n,
                       np, p->d_z, p->g.Lz);
    SPX_CHECK_LAUNCH();
    // continuation + forward z FFT of the 2U profile rows
    const LineFFTHost& f = p->fz;
    const long rows = 2L * U;
    SPX_LAUNCH(with_general, f, k_z_inplace, double, , dim3(unsigned((rows + f.nl - 1) / f.nl)), blk(f),
                  f.lds_bytes(16), p->stream, static_cast<Cd*>(tab), rows, f.dev<Cd>(), np, 1,
                  1, 1.0, p->d_dir, p->g.Cz, p->g.oz);
    SPX_CHECK_LAUNCH();
  }
  SPX_HIP(hipStreamSynchronize(p->stream));
  (void)hipFree(kv);
  p->d_htab = tab;
  p->d_hidx = static_cast<int*>(hid);
  p->nhtab = U;
  return SPX_OK;
}

int project_harmonic(spx_plan* p, void* a, void* b, void* c, void* d, const RkLoad* rk,
                     bool walls_only) {
  const int nz = p->g.nz;
  if (!p->fused_project || !p->d_htab || !p->d_wtop || nz > 64 * 17) return SPX_ERR_UNSUPPORTED;
  const long nlines = p->wlines();
  RkLoad r;
  std::memset(&r, 0, sizeof(r));
  if (rk) r = *rk;
  const double extra = rk ? (rk->nl32 ? 8.0 : 16.0) + 32.0 : 0.0;
  ProfScope ps_(p, rk ? "project_harmonic_rk" : "project_harmonic",
                double(p->wnc()) * (7.0 * 16.0 + extra) + 2.0 * p->nhtab * double(nz) * 16.0);
  const dim3 grid(unsigned((nlines + 3) / 4)), block(256);
  // RK mode of the branch-free variants (lines of at least 64 (KPL - 1) points)
  const int rkm = rk ? (rk->nl32 ? 2 : 1) : 0;
#define SPX_PH(KPL)                                                                            \
  if (nz < 64 * (KPL - 1)) {                                                                   \
    SPX_PH2(KPL, -1);                                                                          \
  } else if (rkm == 0) {                                                                       \
    SPX_PH2(KPL, 0);                                                                           \
  } else if (rkm == 1) {                                                                       \
    SPX_PH2(KPL, 1);                                                                           \
  } else {                                                                                     \
    SPX_PH2(KPL, 2);                                                                           \
  }
#define SPX_PH2(KPL, RKM)                                                                      \
  hipLaunchKernelGGL((k_project_harmonic<KPL, RKM>), grid, block, 0, p->stream, C_<double>(a), \
                     C_<double>(b), C_<double>(c), C_<double>(d), C_<double>(p->bc), nlines,   \
                     nz, p->g.ny, p->d_kx, p->d_ky, p->d_kz,                                   \
                     static_cast<const Cd*>(p->d_wtop), 1.0 / double(nz), r, rk ? 1 : 0,       \
                     walls_only ? C_<double>(p->pw) : nullptr, p->np,                          \
                     static_cast<const Cd*>(p->d_htab), p->d_hidx, p->g.Lz, p->d_khom)
  if (nz <= 64 * 3) {
    SPX_PH2(3, -1);
  } else if (nz <= 64 * 5) {
    SPX_PH(5)
  } else if (nz <= 64 * 9) {
    SPX_PH(9)
  } else {
    SPX_PH(17)
  }
#undef SPX_PH
#undef SPX_PH2
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}

int proj_harmonic(spx_plan* p, void* a, void* b, void* c, int k0, int k1) {
  const long nlines = p->wlines();
  if (p->d_htab) {
    ProfScope ps_(p, "proj_harmonic",
                  6.0 * double(p->wnc()) * 16.0 + 2.0 * p->nhtab * double(p->g.nz) * 16.0);
    hipLaunchKernelGGL(k_proj_harmonic_tab<double>, dim3(unsigned((nlines + 3) / 4)), dim3(256), 0,
                       p->stream, C_<double>(a), C_<double>(b), C_<double>(c),
                       C_<double>(p->bc), static_cast<const Cd*>(p->d_htab), p->d_hidx, nlines,
                       p->g.ny, p->g.nz, p->g.Lz, p->d_khom, p->d_kx, p->d_ky, k0, k1);
    SPX_CHECK_LAUNCH();
    return SPX_OK;
  }
  const LineFFTHost& f = p->fz2;
  const size_t lds = f.lds_bytes(16, 2);
  ProfScope ps_(p, "proj_harmonic", 6.0 * double(p->wnc()) * 16.0);
  SPX_LAUNCH(with_general, f, k_proj_harmonic, double, , dim3(unsigned((nlines + f.nl - 1) / f.nl)), blk(f),
                lds, p->stream, C_<double>(a), C_<double>(b), C_<double>(c), C_<double>(p->bc),
                f.dev<Cd>(), nlines, p->g.ny, p->np, p->g.Lz, p->d_khom, p->d_z, p->d_kx,
                p->d_ky, p->d_dir, p->g.Cz, p->g.oz, k0, k1);
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}

#endif  // SPX_PART 3 (boundary, projection)

#if !defined(SPX_PART) || SPX_PART == 16
int bwall_fused(spx_plan* p, void* a0, void* a1, void* a2, int ncomp, const BWallParams& bp) {
  if (p->g.oz > 16) return fail(SPX_ERR_UNSUPPORTED, "magnetic walls: matching order above 16");
  const LineFFTHost& f = fzt(p, false);
  const long nlines = p->wlines();
  dim3 grid(unsigned((nlines + f.nl - 1) / f.nl), unsigned(ncomp));
  ProfScope ps_(p, "bwall", ncomp * double(p->wnc()) * 2.0 * 16.0);
  SPX_LAUNCH(with_z<16>, f, k_bwall, double, , grid, blk(f), f.lds_bytes(16), p->stream, C_<double>(a0),
                C_<double>(a1), C_<double>(a2), f.dev<Cd>(), nlines, p->np,
                1.0 / double(p->g.nz), bp, p->d_khom, p->d_dir, p->g.Cz, p->g.oz);
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}

int proj_pressure(spx_plan* p, void* d, int k0, int k1) {
  const LineFFTHost& f = fzt(p, false);
  const long nlines = p->wlines();
  ProfScope ps_(p, "proj_pressure", 2.0 * double(p->wnc()) * 16.0);
  const dim3 grid(unsigned((nlines + f.nl - 1) / f.nl));
  const size_t lds = f.lds_bytes(16);
  SPX_LAUNCH(with_z<16>, f, k_proj_pressure, double, , grid, blk(f), lds, p->stream, C_<double>(d),
               C_<double>(p->bc), f.dev<Cd>(), nlines, p->g.ny, 1.0 / double(p->g.nz), p->g.Lz,
               p->d_khom, p->d_z, k0, k1);
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}
#endif  // SPX_PART 16 (magnetic walls, pressure)

#if !defined(SPX_PART) || SPX_PART == 8
static int zline_launch(spx_plan* p, int nterm, const LinComb* lc, const void* const* b, int mode,
                        double* out) {
  if (nterm < 1 || nterm > 3) return fail(SPX_ERR_ARG, "zline_reduce: 1..3 terms");
  const LineFFTHost& fw = fzt(p, false);
  const long nlines = p->wlines();
  const LineFFTHost f = spread(mode == 1 ? fw.with_lines(fw.nl / 2) : fw, nlines, nterm, 1);
  ZTerms<double> d;
  for (int q = 0; q < 3; ++q) {
    const LinComb& c = lc[q < nterm ? q : 0];
    for (int t = 0; t < 3; ++t) {
      d.lc[q].in[t] = static_cast<const Cd*>(c.in[t]);
      d.lc[q].dir[t] = c.dir[t];
      d.lc[q].sgn[t] = c.sgn[t];
    }
    d.b[q] = b ? C_<double>(b[q < nterm ? q : 0]) : nullptr;
  }
  const size_t lds = f.lds_bytes(16, mode == 1 ? 2 : 1) + size_t(f.nl) * f.tpl * sizeof(double);
  ProfScope ps_(p, "zline_reduce", nterm * double(p->wnc()) * 16.0 * (mode == 1 ? 2 : 1));
  SPX_LAUNCH(with_z<16>, f, k_zline_reduce, double, ,
             dim3(unsigned((nlines + f.nl - 1) / f.nl), unsigned(nterm)), blk(f), lds, p->stream, d,
             mode, out, f.dev<Cd>(), nlines, p->g.ny, p->np, p->d_kx, p->d_ky, p->d_kz);
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}

int zline_sumsq(spx_plan* p, int nterm, const LinComb* lc, double* line_out) {
  return zline_launch(p, nterm, lc, nullptr, 0, line_out);
}

int zline_dot(spx_plan* p, int nterm, const LinComb* lc, const void* const* b, double* line_out) {
  return zline_launch(p, nterm, lc, b, 1, line_out);
}

int zline_wall_values(spx_plan* p, const LinComb& lc, double* line_out) {
  return zline_launch(p, 1, &lc, nullptr, 3, line_out);
}

int zline_walls(spx_plan* p, int nterm, const LinComb* lc, double* line_out) {
  return zline_launch(p, nterm, lc, nullptr, 2, line_out);
}

int line_sums(spx_plan* p, int nterm, const double* w, int per, const double* part, double* out) {
  LineWeights lw;
  for (int t = 0; t < 3; ++t) lw.w[t] = t < nterm ? w[t] : 0.0;
  hipLaunchKernelGGL(k_line_sum, dim3(unsigned(p->mem), unsigned(per)), dim3(1024), 0, p->stream,
                     part, lw, nterm, per, p->wlines() / p->mem, p->g.ny, out);
  SPX_CHECK_LAUNCH();
  return SPX_OK;
}
#endif  // SPX_PART 8 (diagnostics)

}  // namespace spx

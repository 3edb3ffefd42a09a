// Device-side FFT building blocks for the fluidsim_amd engine (gfx950).
//
// Complex numbers are interleaved (re, im) pairs of T (float or double), the
// layout numpy's complex64/complex128 use, so K arrays cross the C-ABI as
// plain pointers.
//
// Transforms are Stockham autosort FFTs.  Power-of-two lengths run radix-2 to
// radix-16 stages: in the strided passes the plan of TilePlan (fsx_tile.h), in
// the LDS row pass radix 8 while at least three factors of two remain, then 4
// or 2.  Other lengths: mixed radix, below.  Butterfly j of a stage with sub-transform length Ns reads positions
// j + r N/R, multiplies input r by W_{Ns R}^{r k} (k = j mod Ns), applies a
// hard-coded DFT_R and writes output r to (j - k) R + k + r Ns, so the
// result is in natural order without a bit-reversal pass.
//
// The strided passes of power-of-two lengths keep the first stage in registers
// (inputs come straight from HBM) and the last stage in registers (outputs go
// straight to HBM: for the last stage k = j, so output r lands at position
// j + r Ns); LDS holds only what one stage hands to the next.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace fsx {

template <typename T>
struct cpx {
  T x, y;
};

template <typename T>
__device__ __forceinline__ cpx<T> mk(T a, T b) {
  cpx<T> r;
  r.x = a;
  r.y = b;
  return r;
}
template <typename T>
__device__ __forceinline__ cpx<T> operator+(cpx<T> a, cpx<T> b) {
  return mk<T>(a.x + b.x, a.y + b.y);
}
template <typename T>
__device__ __forceinline__ cpx<T> operator-(cpx<T> a, cpx<T> b) {
  return mk<T>(a.x - b.x, a.y - b.y);
}
template <typename T>
__device__ __forceinline__ cpx<T> operator*(cpx<T> a, cpx<T> b) {
  return mk<T>(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
template <typename T>
__device__ __forceinline__ cpx<T> scale(cpx<T> a, T s) {
  return mk<T>(a.x * s, a.y * s);
}
// scale whose products are not fused into later additions
template <typename T>
__device__ __forceinline__ cpx<T> scale_rounded(cpx<T> a, T s) {
#pragma clang fp contract(off)
  return mk<T>(a.x * s, a.y * s);
}
template <typename T>
__device__ __forceinline__ cpx<T> conj(cpx<T> a) {
  return mk<T>(a.x, -a.y);
}
// multiply by i
template <typename T>
__device__ __forceinline__ cpx<T> mul_i(cpx<T> a) {
  return mk<T>(-a.y, a.x);
}
template <typename T>
__device__ __forceinline__ cpx<T> zero() {
  return mk<T>(T(0), T(0));
}

// a b + c with one rounding, whatever the fp contraction setting
template <typename T>
__device__ __forceinline__ T fma_t(T a, T b, T c) {
  if constexpr (sizeof(T) == 4)
    return __builtin_fmaf(a, b, c);
  else
    return __builtin_fma(a, b, c);
}

// DIR = -1: forward transform, kernel exp(-2 pi i jk/N).
// DIR = +1: inverse transform, kernel exp(+2 pi i jk/N).
// Multiplication by exp(DIR * i pi / 2): forward -> -i, inverse -> +i.
template <typename T, int DIR>
__device__ __forceinline__ cpx<T> rot90(cpx<T> a) {
  return DIR < 0 ? mk<T>(a.y, -a.x) : mk<T>(-a.y, a.x);
}

template <typename T, int DIR>
__device__ __forceinline__ void dft2(cpx<T>* v) {
  cpx<T> a = v[0], b = v[1];
  v[0] = a + b;
  v[1] = a - b;
}

template <typename T, int DIR>
__device__ __forceinline__ void dft4(cpx<T>* v) {
  cpx<T> t0 = v[0] + v[2], t1 = v[0] - v[2];
  cpx<T> t2 = v[1] + v[3], t3 = rot90<T, DIR>(v[1] - v[3]);
  v[0] = t0 + t2;
  v[2] = t0 - t2;
  v[1] = t1 + t3;
  v[3] = t1 - t3;
}

// 8-point DFT as one radix-2 step (stride 4) followed by two 4-point DFTs:
// X[2m] = DFT4(a[k] + a[k+4]), X[2m+1] = DFT4((a[k] - a[k+4]) w8^k).  The
// factor 1/sqrt 2 of w8 and w8^3 is folded into the last additions as fused
// multiply-adds (52 instead of 56 operations).
template <typename T, int DIR>
__device__ __forceinline__ void dft8(cpx<T>* v) {
  const T h = T(0.70710678118654752440084436210484903928);
  cpx<T> b[4], c[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    b[k] = v[k] + v[k + 4];
    c[k] = v[k] - v[k + 4];
  }
  dft4<T, DIR>(b);
  // sqrt 2 w8 c1 and sqrt 2 w8^3 c3
  const cpx<T> p = DIR < 0 ? mk<T>(c[1].x + c[1].y, c[1].y - c[1].x)
                           : mk<T>(c[1].x - c[1].y, c[1].x + c[1].y);
  const cpx<T> q = DIR < 0 ? mk<T>(c[3].y - c[3].x, -(c[3].x + c[3].y))
                           : mk<T>(-(c[3].x + c[3].y), c[3].x - c[3].y);
  c[2] = rot90<T, DIR>(c[2]);
  const cpx<T> t0 = c[0] + c[2], t1 = c[0] - c[2];
  const cpx<T> u = p + q, w = rot90<T, DIR>(p - q);
  v[0] = b[0];
  v[2] = b[1];
  v[4] = b[2];
  v[6] = b[3];
  v[1] = mk<T>(fma_t(h, u.x, t0.x), fma_t(h, u.y, t0.y));
  v[5] = mk<T>(fma_t(-h, u.x, t0.x), fma_t(-h, u.y, t0.y));
  v[3] = mk<T>(fma_t(h, w.x, t1.x), fma_t(h, w.y, t1.y));
  v[7] = mk<T>(fma_t(-h, w.x, t1.x), fma_t(-h, w.y, t1.y));
}

// a exp(DIR 2 pi i m / 16) for a constant m
template <typename T, int DIR, int M>
__device__ __forceinline__ cpx<T> w16(cpx<T> a) {
  constexpr int m = M & 15;
  if constexpr (m == 0) {
    return a;
  } else if constexpr (m == 4) {
    return rot90<T, DIR>(a);
  } else {
    // cos and sin of 2 pi m / 16 from the first-octant values
    constexpr T c1 = T(0.92387953251128675612818318939678828682);  // cos(pi/8)
    constexpr T s1 = T(0.38268343236508977172845998403039886676);  // sin(pi/8)
    constexpr T h = T(0.70710678118654752440084436210484903928);
    constexpr T ct[16] = {T(1), c1, h, s1, T(0), -s1, -h, -c1, T(-1), -c1, -h, -s1, T(0), s1, h, c1};
    constexpr T c = ct[m], sn = ct[(m + 12) & 15];  // sin x = cos(x - pi/2)
    const T wi = DIR < 0 ? -sn : sn;
    // explicit fused multiply-adds: the rounding is then the same in every
    // pass that inlines this (no choice left to fp contraction)
    return mk<T>(fma_t(a.x, c, -(a.y * wi)), fma_t(a.x, wi, a.y * c));
  }
}

// 16-point DFT as 4 x 4: with n = 4 n1 + n2 and k = k1 + 4 k2,
// X[k1 + 4 k2] = DFT4_{n2}( W16^{n2 k1} DFT4_{n1}(x[4 n1 + n2])[k1] )[k2].
template <typename T, int DIR>
__device__ __forceinline__ void dft16(cpx<T>* v) {
  cpx<T> y[4][4];
#pragma unroll
  for (int n2 = 0; n2 < 4; ++n2) {
#pragma unroll
    for (int n1 = 0; n1 < 4; ++n1) y[n2][n1] = v[4 * n1 + n2];
    dft4<T, DIR>(y[n2]);
  }
  y[1][1] = w16<T, DIR, 1>(y[1][1]);
  y[1][2] = w16<T, DIR, 2>(y[1][2]);
  y[1][3] = w16<T, DIR, 3>(y[1][3]);
  y[2][1] = w16<T, DIR, 2>(y[2][1]);
  y[2][2] = w16<T, DIR, 4>(y[2][2]);
  y[2][3] = w16<T, DIR, 6>(y[2][3]);
  y[3][1] = w16<T, DIR, 3>(y[3][1]);
  y[3][2] = w16<T, DIR, 6>(y[3][2]);
  y[3][3] = w16<T, DIR, 9>(y[3][3]);
#pragma unroll
  for (int k1 = 0; k1 < 4; ++k1) {
    cpx<T> b[4] = {y[0][k1], y[1][k1], y[2][k1], y[3][k1]};
    dft4<T, DIR>(b);
#pragma unroll
    for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = b[k2];
  }
}

template <typename T, int DIR, int R>
__device__ __forceinline__ void dftR(cpx<T>* v) {
  static_assert(R == 16 || R == 8 || R == 4 || R == 2, "radix 2, 4, 8 or 16");
  if constexpr (R == 16)
    dft16<T, DIR>(v);
  else if constexpr (R == 8)
    dft8<T, DIR>(v);
  else if constexpr (R == 4)
    dft4<T, DIR>(v);
  else
    dft2<T, DIR>(v);
}

// 3-point DFT: y0 = a + b + c, y1,2 = a - (b + c)/2 +- i DIR (sqrt 3 / 2)(b - c).
template <typename T, int DIR>
__device__ __forceinline__ void dft3(cpx<T>* v) {
  const T h = T(0.86602540378443864676372317075293618347);
  const cpx<T> s = v[1] + v[2];
  const cpx<T> t = v[0] - scale(s, T(0.5));
  const cpx<T> u = rot90<T, DIR>(scale(v[1] - v[2], h));
  v[0] = v[0] + s;
  v[1] = t + u;
  v[2] = t - u;
}

// 5-point DFT from the cosines and sines of 2 pi / 5 and 4 pi / 5:
// y1,4 = x0 + c1 a1 + c2 a2 +- i DIR (s1 b1 + s2 b2),
// y2,3 = x0 + c2 a1 + c1 a2 +- i DIR (s2 b1 - s1 b2),
// a1 = x1 + x4, a2 = x2 + x3, b1 = x1 - x4, b2 = x2 - x3.
template <typename T, int DIR>
__device__ __forceinline__ void dft5(cpx<T>* v) {
  const T c1 = T(0.30901699437494742410229341718281905886);
  const T c2 = T(-0.80901699437494742410229341718281905886);
  const T s1 = T(0.95105651629515357211643933337938214340);
  const T s2 = T(0.58778525229247312916870595463907276860);
  const cpx<T> a1 = v[1] + v[4], a2 = v[2] + v[3];
  const cpx<T> b1 = v[1] - v[4], b2 = v[2] - v[3];
  const cpx<T> t1 = v[0] + scale(a1, c1) + scale(a2, c2);
  const cpx<T> t2 = v[0] + scale(a1, c2) + scale(a2, c1);
  const cpx<T> u1 = rot90<T, DIR>(scale(b1, s1) + scale(b2, s2));
  const cpx<T> u2 = rot90<T, DIR>(scale(b1, s2) - scale(b2, s1));
  v[0] = v[0] + a1 + a2;
  v[1] = t1 + u1;
  v[4] = t1 - u1;
  v[2] = t2 + u2;
  v[3] = t2 - u2;
}

// Radix of stage s of a length-2^logN transform (8s first, then 4 or 2).
__host__ __device__ __forceinline__ int stage_log_radix(int logN, int logNs) {
  const int rem = logN - logNs;
  return rem >= 3 ? 3 : rem;
}

// LDS address with one pad slot per 32 elements: power-of-two strides of
// the Stockham write patterns then fall on different banks.
__device__ __forceinline__ int lpad(int a) { return a + (a >> 5); }

// Apply the Stockham twiddles W_{Ns R}^{r k} to v[1..R-1].
// tw is a table exp(-2 pi i m / Ntab) with Ntab = N << twshift.
template <typename T, int DIR, int R, int LOGR>
__device__ __forceinline__ void twiddle(cpx<T>* v, int k, int logN, int logNs,
                                        const cpx<T>* tw, int twshift) {
  const int sh = (logN - logNs - LOGR) + twshift;
#pragma unroll
  for (int r = 1; r < R; ++r) {
    cpx<T> w = tw[(r * k) << sh];
    if (DIR > 0) w.y = -w.y;
    v[r] = v[r] * w;
  }
}

// Full in-LDS FFT over `lines` rows stored at buf[line * ldr + lpad(pos)]
// (row layout, butterfly-fast thread map), all stages.  Used by the row
// (x) pass.  Caller synchronises before the call.
template <typename T, int DIR, int EPT, int R, int kT>
__device__ __forceinline__ void lds_stage_rows(cpx<T>* buf, int logN,
                                               int logNs, int lines, int ldr,
                                               const cpx<T>* tw, int twshift) {
  constexpr int LOGR = R == 8 ? 3 : (R == 4 ? 2 : 1);
  constexpr int NB = EPT / R;
  const int lognb = logN - LOGR;
  const int total = lines << lognb;
  const int Ns = 1 << logNs;
  cpx<T> v[NB][R];
  int ob[NB], op[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int b = threadIdx.x + i * kT;
    if (b < total) {
      const int j = b & ((1 << lognb) - 1);
      const int line = b >> lognb;
      const int k = j & (Ns - 1);
      const cpx<T>* row = buf + line * ldr;
#pragma unroll
      for (int r = 0; r < R; ++r) v[i][r] = row[lpad(j + (r << lognb))];
      if (logNs > 0) twiddle<T, DIR, R, LOGR>(v[i], k, logN, logNs, tw, twshift);
      dftR<T, DIR, R>(v[i]);
      ob[i] = line * ldr;
      op[i] = ((j - k) << LOGR) + k;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int b = threadIdx.x + i * kT;
    if (b < total) {
#pragma unroll
      for (int r = 0; r < R; ++r) buf[ob[i] + lpad(op[i] + r * Ns)] = v[i][r];
    }
  }
  __syncthreads();
}

template <typename T, int DIR, int EPT, int kT>
__device__ __forceinline__ void lds_fft_rows(cpx<T>* buf, int logN, int lines,
                                             int ldr, const cpx<T>* tw,
                                             int twshift) {
  int logNs = 0;
  while (logNs < logN) {
    const int lr = stage_log_radix(logN, logNs);
    if (lr == 3)
      lds_stage_rows<T, DIR, EPT, 8, kT>(buf, logN, logNs, lines, ldr, tw, twshift);
    else if (lr == 2)
      lds_stage_rows<T, DIR, EPT, 4, kT>(buf, logN, logNs, lines, ldr, tw, twshift);
    else
      lds_stage_rows<T, DIR, EPT, 2, kT>(buf, logN, logNs, lines, ldr, tw, twshift);
    logNs += lr;
  }
}

// ------------------------------------------------------ mixed-radix lengths
// Transforms of any length N (grids that are not powers of two) run as
// Stockham stages whose radix is one of 2 .. 13, 15 or 16 (products of two
// coprime factors by the prime-factor index maps, without twiddles; 7, 11 and
// 13 from the symmetric sums and differences of their inputs) or, for any
// other prime, a direct DFT, with the same index rule as the power-of-two
// stages: butterfly j (k = j mod Ns) reads positions j + r N/R, applies
// W_{Ns R}^{r k} and DFT_R, and writes output r to (j - k) R + k + r Ns.
// gen_factor picks the fewest stages (240 = 16 15, 192 = 16 12, 160 = 16 10):
// what a stage costs is its LDS round trip and its barriers.  A thread holds
// its butterflies (up to kGenRegs values) across the barrier between reading
// and writing, so a tile that fits the registers needs one LDS buffer; tiles
// beyond that, and direct stages, read one buffer and write a second.
//
// ns3d 240 x 192 x 160 FP64, per stage: rows 1035 -> 270 us, y-inverse 151 ->
// 160, curl 250 -> 148, z-forward + RK 279 -> 154 us (y-passes and rows of the
// new figures from 4 overlapping chunks), against radices of at most 8, index
// divisions per element, full-length transforms of the real rows and loads
// one at a time.
constexpr int kMaxStages = 16;
constexpr int kGenRegs = 16;

// Values of a thread's butterflies in a stage of radix r.
constexpr int gen_held(int r) { return r * (kGenRegs / r); }

// Whether tiles of n elements run in one buffer with kT threads.
inline bool gen_in_place(const int* rad, int nst, long long n, int kT) {
  for (int i = 0; i < nst; ++i)
    if (rad[i] > kGenRegs || n > (long long)kT * gen_held(rad[i])) return false;
  return true;
}

// Element (line, pos) of a tile in LDS: line sl + pos sp (strided passes:
// sl = 1, sp = lines | 1; row passes: sl = row stride, sp = 1).
struct TileLayout {
  int sl, sp;
  __device__ __forceinline__ int at(int line, int pos) const { return line * sl + pos * sp; }
};

// n / d for 0 <= n, n d < 2^32, with m = magic_of(d); d = 1 has no magic
__device__ __forceinline__ unsigned magic_of(unsigned d) { return 0xffffffffu / d + 1u; }
__device__ __forceinline__ int magic_div(int n, unsigned m, int d) {
  return d == 1 ? n : (int)__umulhi((unsigned)n, m);
}

// Index with k mod A = k1 and k mod B = k2 (A, B coprime).
constexpr int crt_index(int A, int B, int k1, int k2) {
  for (int k = 0; k < A * B; ++k)
    if (k % A == k1 && k % B == k2) return k;
  return 0;
}

// P-point DFT of an odd prime: with a_m = x_m + x_{P-m}, b_m = x_m - x_{P-m},
// X_r, X_{P-r} = x_0 + sum_m c_{mr} a_m +- i DIR sum_m s_{mr} b_m.
template <int P>
struct PrimeTab;
template <>
struct PrimeTab<7> {
  static constexpr double c[4] = {1, 0.62348980185873353052500488400424, -0.22252093395631440428890256449679,
                                  -0.90096886790241912623610231950745};
  static constexpr double s[4] = {0, 0.78183148246802980870844452667406, 0.97492791218182360701813168299393,
                                  0.43388373911755812047576833284836};
};
template <>
struct PrimeTab<11> {
  static constexpr double c[6] = {1, 0.84125353283118116886181164891937, 0.41541501300188642552927414922962,
                                  -0.14231483827328514044379266861637, -0.65486073394528506405692507246629,
                                  -0.95949297361449738989036805706633};
  static constexpr double s[6] = {0, 0.54064081745559758210763595431869, 0.90963199535451837141171538307903,
                                  0.98982144188093273237609203777872, 0.75574957435425828377403584397234,
                                  0.28173255684142969771141791534662};
};
template <>
struct PrimeTab<13> {
  static constexpr double c[7] = {1, 0.88545602565320989590037552201510, 0.56806474673115580251180755912752,
                                  0.12053668025532305334906768745254, -0.35460488704253562596963789260002,
                                  -0.74851074817110109863463059970135, -0.97094181742605202715698227629379};
  static constexpr double s[7] = {0, 0.46472317204376854565601533513310, 0.82298386589365639457961742343938,
                                  0.99270887409805399280075164949252, 0.93501624268541482343978459983783,
                                  0.66312265824079520237678549266769, 0.23931566428755776714875372626021};
};

template <typename T, int DIR, int P>
__device__ __forceinline__ void dft_prime(cpx<T>* v) {
  constexpr int H = (P - 1) / 2;
  cpx<T> a[H + 1], b[H + 1];
#pragma unroll
  for (int m = 1; m <= H; ++m) {
    a[m] = v[m] + v[P - m];
    b[m] = v[m] - v[P - m];
  }
  const cpx<T> x0 = v[0];
#pragma unroll
  for (int m = 1; m <= H; ++m) v[0] = v[0] + a[m];
#pragma unroll
  for (int r = 1; r <= H; ++r) {
    cpx<T> t = x0, u = zero<T>();
#pragma unroll
    for (int m = 1; m <= H; ++m) {
      const int q = (m * r) % P, qs = q <= H ? q : P - q;
      const T c = T(PrimeTab<P>::c[qs]), s = T(q <= H ? PrimeTab<P>::s[qs] : -PrimeTab<P>::s[qs]);
      t = mk<T>(fma_t(c, a[m].x, t.x), fma_t(c, a[m].y, t.y));
      u = mk<T>(fma_t(s, b[m].x, u.x), fma_t(s, b[m].y, u.y));
    }
    u = rot90<T, DIR>(u);
    v[r] = t + u;
    v[P - r] = t - u;
  }
}

// 9-point DFT as 3 x 3 (n = 3 n1 + n2, k = k1 + 3 k2) with W9^{n2 k1} between.
template <typename T, int DIR>
__device__ __forceinline__ void dft9(cpx<T>* v) {
  constexpr T c1 = T(0.76604444311897803520239265055542), s1 = T(0.64278760968653932632264340990726);
  constexpr T c2 = T(0.17364817766693034885171662676931), s2 = T(0.98480775301220805936674302458952);
  constexpr T c4 = T(-0.93969262078590838405410927732473), s4 = T(0.34202014332566873304409961468226);
  cpx<T> y[3][3];
#pragma unroll
  for (int n2 = 0; n2 < 3; ++n2) {
#pragma unroll
    for (int n1 = 0; n1 < 3; ++n1) y[n2][n1] = v[3 * n1 + n2];
    dft3<T, DIR>(y[n2]);
  }
  auto tw = [](cpx<T> x, T c, T s) {
    const T w = DIR < 0 ? -s : s;
    return mk<T>(fma_t(x.x, c, -(x.y * w)), fma_t(x.x, w, x.y * c));
  };
  y[1][1] = tw(y[1][1], c1, s1);
  y[1][2] = tw(y[1][2], c2, s2);
  y[2][1] = tw(y[2][1], c2, s2);
  y[2][2] = tw(y[2][2], c4, s4);
#pragma unroll
  for (int k1 = 0; k1 < 3; ++k1) {
    cpx<T> b[3] = {y[0][k1], y[1][k1], y[2][k1]};
    dft3<T, DIR>(b);
#pragma unroll
    for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = b[k2];
  }
}

template <typename T, int DIR, int R>
__device__ __forceinline__ void dft_any(cpx<T>* v);

// A B-point DFT of coprime A, B (prime-factor maps): n = B n1 + A n2, output
// k = k1 mod A = k2 mod B; no twiddles between the two.
template <typename T, int DIR, int A, int B>
__device__ __forceinline__ void dft_pf(cpx<T>* v) {
  cpx<T> y[A][B];
#pragma unroll
  for (int n2 = 0; n2 < B; ++n2) {
    cpx<T> a[A];
#pragma unroll
    for (int n1 = 0; n1 < A; ++n1) a[n1] = v[(B * n1 + A * n2) % (A * B)];
    dft_any<T, DIR, A>(a);
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) y[k1][n2] = a[k1];
  }
#pragma unroll
  for (int k1 = 0; k1 < A; ++k1) {
    dft_any<T, DIR, B>(y[k1]);
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) v[crt_index(A, B, k1, k2)] = y[k1][k2];
  }
}

template <typename T, int DIR, int R>
__device__ __forceinline__ void dft_any(cpx<T>* v) {
  if constexpr (R == 3)
    dft3<T, DIR>(v);
  else if constexpr (R == 5)
    dft5<T, DIR>(v);
  else if constexpr (R == 6)
    dft_pf<T, DIR, 2, 3>(v);
  else if constexpr (R == 7 || R == 11 || R == 13)
    dft_prime<T, DIR, R>(v);
  else if constexpr (R == 9)
    dft9<T, DIR>(v);
  else if constexpr (R == 10)
    dft_pf<T, DIR, 2, 5>(v);
  else if constexpr (R == 12)
    dft_pf<T, DIR, 4, 3>(v);
  else if constexpr (R == 15)
    dft_pf<T, DIR, 3, 5>(v);
  else
    dftR<T, DIR, R>(v);
}

// One stage of radix R over `lines` lines: A -> B (the same buffer where the
// butterflies of all threads fit their registers).  The twiddles are entries
// of tw[m] = exp(-2 pi i m / (N tws)).
struct GenStage {
  int N, Ns, lines, logL;  // logL >= 0: line-fast thread map, lines = 2^logL
  int tws;
};
template <typename T, int DIR, int R, int kT>
__device__ __forceinline__ void gen_stage(const cpx<T>* A, cpx<T>* B, const TileLayout& lay,
                                          const cpx<T>* tw, const GenStage& g) {
  constexpr int NB = kGenRegs / R;
  const int NR = g.N / R, Ns = g.Ns;
  const int nb = NR * g.lines, step = NR / Ns * g.tws;
  const unsigned mNs = magic_of(Ns), mNR = magic_of(NR);
  // (one turn where A is B)
  for (int b0 = threadIdx.x; b0 < nb + (int)threadIdx.x; b0 += NB * kT) {
    cpx<T> v[NB][R];
    int o[NB], ks[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int b = b0 + i * kT;
      if (i > 0 && b >= nb) break;
      int line, j;
      if (g.logL >= 0) {
        line = b & (g.lines - 1);
        j = b >> g.logL;
      } else {
        line = magic_div(b, mNR, NR);
        j = b - line * NR;
      }
      const int k = j - magic_div(j, mNs, Ns) * Ns;
      ks[i] = k * step;
      o[i] = lay.at(line, (j - k) * R + k);
      if (b < nb) {
        const cpx<T>* a = A + lay.at(line, j);
#pragma unroll
        for (int r = 0; r < R; ++r) v[i][r] = a[r * NR * lay.sp];
        if (Ns > 1) {
#pragma unroll
          for (int r = 1; r < R; ++r) {
            cpx<T> w = tw[r * ks[i]];
            if (DIR > 0) w.y = -w.y;
            v[i][r] = v[i][r] * w;
          }
        }
        dft_any<T, DIR, R>(v[i]);
      }
    }
    if (A == B) __syncthreads();
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int b = b0 + i * kT;
      if (b < nb) {
#pragma unroll
        for (int r = 0; r < R; ++r) B[o[i] + r * Ns * lay.sp] = v[i][r];
      }
    }
  }
}

// Direct DFT of a prime radix R without a dedicated butterfly: output r of
// butterfly j is sum_m (x_m W_{Ns R}^{m k}) W_R^{m r}.
template <typename T, int DIR, int kT>
__device__ __forceinline__ void gen_direct(const cpx<T>* A, cpx<T>* B, const TileLayout& lay,
                                           const cpx<T>* tw, const GenStage& g, int R) {
  const int NR = g.N / R, Ns = g.Ns;
  const int nb = NR * g.lines, step = NR / Ns;
  for (int b = threadIdx.x; b < nb; b += kT) {
    const int line = g.logL >= 0 ? b & (g.lines - 1) : b / NR;
    const int j = g.logL >= 0 ? b >> g.logL : b - line * NR;
    const int k = j % Ns;
    const int o = (j - k) * R + k;
    for (int r = 0; r < R; ++r) {
      cpx<T> acc = zero<T>();
      int q = 0;  // m r mod R
      for (int m = 0; m < R; ++m) {
        cpx<T> w = tw[m * k * step * g.tws];
        cpx<T> u = tw[q * NR * g.tws];
        if (DIR > 0) {
          w.y = -w.y;
          u.y = -u.y;
        }
        acc = acc + (A[lay.at(line, j + m * NR)] * w) * u;
        q += r;
        if (q >= R) q -= R;
      }
      B[lay.at(line, o + r * Ns)] = acc;
    }
  }
}

// All stages of `lines` transforms of length N over the tile in A (B: the
// second buffer, or A), kT threads.  The caller synchronises before; returns the
// buffer that holds the result, after a barrier.
template <typename T, int DIR, int kT>
__device__ __forceinline__ cpx<T>* gen_fft(cpx<T>* A, cpx<T>* B, const TileLayout& layout,
                                           const cpx<T>* tw, int tws, int N, int lines, int logL,
                                           int nst, const int* rad) {
  int Ns = 1;
  for (int s = 0; s < nst; ++s) {
    const int R = rad[s];
    // opaque to the optimizer: the strides of every radix below would
    // otherwise be computed ahead of the loop and kept in registers
    int n = __builtin_amdgcn_readfirstlane(N), sp = __builtin_amdgcn_readfirstlane(layout.sp);
    asm volatile("" : "+s"(n), "+s"(sp));
    const TileLayout lay{layout.sl, __builtin_amdgcn_readfirstlane(sp)};
    const GenStage g{__builtin_amdgcn_readfirstlane(n), Ns, lines, logL, tws};
    switch (R) {
#define FSX_GEN_RADIX(r) \
  case r: gen_stage<T, DIR, r, kT>(A, B, lay, tw, g); break;
      FSX_GEN_RADIX(2)
      FSX_GEN_RADIX(3)
      FSX_GEN_RADIX(4)
      FSX_GEN_RADIX(5)
      FSX_GEN_RADIX(6)
      FSX_GEN_RADIX(7)
      FSX_GEN_RADIX(8)
      FSX_GEN_RADIX(9)
      FSX_GEN_RADIX(10)
      FSX_GEN_RADIX(11)
      FSX_GEN_RADIX(12)
      FSX_GEN_RADIX(13)
      FSX_GEN_RADIX(15)
      FSX_GEN_RADIX(16)
#undef FSX_GEN_RADIX
      default: gen_direct<T, DIR, kT>(A, B, lay, tw, g, R); break;
    }
    __syncthreads();
    cpx<T>* t = A;
    A = B;
    B = t;
    Ns *= R;
  }
  return A;
}

// Stage radices of a length-n transform (host): the fewest stages of the
// butterflies above, the most even of those (smallest sum of radices), larger
// radices first; other primes are stages of their own.  Returns the number
// of stages, or -1 when more than kMaxStages would be needed.
inline void gen_split(int n, int maxr, int* cur, int nc, int sum, int* best, int& nbest,
                      int& sbest) {
  if (n == 1) {
    if (nc < nbest || (nc == nbest && sum < sbest)) {
      nbest = nc;
      sbest = sum;
      for (int i = 0; i < nc; ++i) best[i] = cur[i];
    }
    return;
  }
  if (nc >= nbest) return;
  for (int r = maxr; r >= 2; --r) {
    if (r == 14 || n % r != 0) continue;
    cur[nc] = r;
    gen_split(n / r, r, cur, nc + 1, sum + r, best, nbest, sbest);
  }
}
inline int gen_factor(int n, int* rad) {
  // primes without a butterfly
  int big[kMaxStages], nbig = 0, m = n;
  for (int p : {2, 3, 5, 7, 11, 13})
    while (m % p == 0) m /= p;
  int smooth = n / m;
  for (int p = 17; m > 1; p += 2) {
    if ((long long)p * p > m) p = m;
    while (m % p == 0) {
      if (nbig >= kMaxStages) return -1;
      big[nbig++] = p;
      m /= p;
    }
  }
  int cur[kMaxStages + 1], best[kMaxStages + 1];
  int nbest = kMaxStages + 1, sbest = 0;
  gen_split(smooth, 16, cur, 0, 0, best, nbest, sbest);
  if (nbest + nbig > kMaxStages) return -1;
  int ns = 0;
  for (int i = 0; i < nbest; ++i) rad[ns++] = best[i];
  for (int i = 0; i < nbig; ++i) rad[ns++] = big[i];
  return ns;
}

// Kept-index map of a signed (y or z) wavenumber axis: kept indices are
// [0, lo) U [n - hi, n); compact index j in [0, lo + hi).
struct AxisMap {
  int n, lo, hi;
  __host__ __device__ int nk() const { return lo + hi; }
  __host__ __device__ int full(int j) const {
    return j < lo ? j : j + (n - lo - hi);
  }
  __host__ __device__ int compact(int i) const {
    return i < lo ? i : (i >= n - hi ? i - (n - lo - hi) : -1);
  }
};

// Signed wavenumber index with the Nyquist index mapped to +n/2.
__host__ __device__ __forceinline__ int ksigned(int i, int n) {
  return i <= n / 2 ? i : i - n;
}

}  // namespace fsx

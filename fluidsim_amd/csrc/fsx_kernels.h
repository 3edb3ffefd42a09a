// Pass kernels of the fluidsim_amd engine.
//
// Array layouts in HBM (C order, complex = interleaved re/im):
//   X  (physical)     : (nz, ny, nx) real            (2D: nz = 1)
//   K  (spectral)     : (nz, ny, nkx) complex, nkx = nx/2 + 1
//   W1 (after z-pass) : (nz, nyk, ld1) complex       (3D only)
//   W2 (after y-pass) : (nz, ny,  ld2) complex
// mx is the number of kept kx indices and nyk the number of kept ky indices
// of the pass (everything for plain transforms, the bounding box of the
// non-dealiased modes for the solver passes, whose pruned modes are zero and
// are neither loaded nor stored).  ld1, ld2 >= mx are row strides rounded up
// to 128 bytes so that every run of a tile starts on a cache line.
//
// A strided pass transforms along y or z: a workgroup owns L adjacent lines
// (consecutive kx, the contiguous index) of length N, so every global access
// is a contiguous run of L complex numbers.  The first Stockham stage reads
// its butterfly inputs straight from HBM into registers, the middle stages
// go through LDS, the last stage writes straight to HBM.  A row pass
// transforms along x (real <-> half complex through a complex FFT of length
// nx/2) and is where the physical-space products are fused.
#pragma once

#include <algorithm>

#include "fsx_fft.h"
#include "fsx_pointwise.h"
#include "fsx_tile.h"

namespace fsx {

// ---------------------------------------------------------------- strided
// Workgroups are dispatched round-robin over the XCDs (workgroup b runs on
// XCD b mod kNXCD), each XCD with its own L2.  In passes over K rows
// (nkx = nx/2 + 1 complex values, not line-aligned), and in passes whose
// tiles hold runs shorter than a 128-byte line (long transforms leave few
// lines per tile), neighbouring line chunks share cache lines, so there
// consecutive tiles are given to the same XCD: XCD x takes the x-th
// contiguous range.
constexpr int kNXCD = 8;
__device__ __forceinline__ int xcd_remap(int b, int nb) {
  if (nb < kNXCD) return b;
  const int x = b % kNXCD, local = b / kNXCD;
  const int q = nb / kNXCD, rem = nb % kNXCD;
  return x < rem ? x * (q + 1) + local : rem * (q + 1) + (x - rem) * q + local;
}

// Strided pass.  LOGN > 0: length 2^LOGN, N L / 2^LOGE threads (4 L lines
// where the op stacks its outputs); LOGN = 0: any length, kGenThr threads.
template <typename T, int DIR, int LOGN, int LOGE, class Op>
// (mixed radix: at least 4, FP64 3, or 2 where transforms are kept, waves per SIMD; the
// widest of the many butterflies would take 200 to 500 registers otherwise)
static __global__ __launch_bounds__((LOGN > 0 ? strided_threads<T, Op>(LOGN, LOGE) : kGenThr),
                                    (LOGN > 0 ? 1 : (Op::kMulti ? 2 : (sizeof(T) == 8 ? 3 : 4))))
void k_strided(Op op) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const StridedDesc<T>& d = op.d;
  cpx<T>* s_tw = reinterpret_cast<cpx<T>*>(smem_raw);
  cpx<T>* buf;
  // (tile_fft's first barrier precedes every twiddle read)
  if constexpr (LOGN > 0) {
    buf = s_tw + TilePlan<LOGN, LOGE>::NTW;
    tile_twiddles<T, LOGN, LOGE>(s_tw, d.tw);
  } else {
    buf = s_tw + d.N;
    for (int i = threadIdx.x; i < d.N; i += kGenThr) s_tw[i] = d.tw[i];
  }
  const int nchunks = (d.nlines + d.L - 1) >> d.logL;
  const int b = d.kio ? xcd_remap(blockIdx.x, gridDim.x) : (int)blockIdx.x;
  const int o = b / nchunks;
  const int line0 = (b - o * nchunks) << d.logL;
  op.template run<DIR, LOGN, LOGE>(buf, s_tw, o, line0);
}

// An op's pitch() is the larger stride of its two sides (elements between
// neighbouring positions), for the launcher's check of the lanes' reach.
//
// Plain pass: one field per workgroup (blockIdx.y).  The op names the two
// sides of field f, plane o: geometry (in_lines, out_lines) and base
// pointers of line line0 (in_base, out_base).
template <typename T, class Self>
struct PlainRun {
  static constexpr bool kMulti = false;
  static constexpr bool kFieldPerBlock = true;
  template <int DIR, int LOGN, int LOGE>
  __device__ __forceinline__ void run(cpx<T>* buf, const cpx<T>* tw, int o, int line0) const {
    const Self& s = static_cast<const Self&>(*this);
    const int nl = s.d.nlines - line0, f = blockIdx.y;
    const Lines gi = s.in_lines(nl), go = s.out_lines(nl);
    const cpx<T>* in = s.in + f * s.ifs + s.in_plane(o) + line0;
    cpx<T>* out = s.out + f * s.ofs + s.out_plane(o) + line0;
    const unsigned char* mask = s.mask ? s.mask + s.out_plane(o) + line0 : nullptr;
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, s.d, s.d.logL, [&](const Slot& t) { return ln_load<LOGN, T>(gi, in, t); },
        [&](const Slot& t, cpx<T> v) {
          if (ln_masked<LOGN>(go, mask, t)) v = zero<T>();
          ln_store<LOGN, T>(go, out, t, v);
        });
  }
};

// Plain z-pass, inverse: K (nz, ny, nkx) -> W1 (nz, nyk, ld1).
// Lines are kx in [0, mx); planes are the kept ky rows.
template <typename T>
struct OpZInv : PlainRun<T, OpZInv<T>> {
  StridedDesc<T> d;
  const cpx<T>* in;
  cpx<T>* out;
  long long ifs, ofs;  // field strides (elements)
  int ny, nkx, ld1;
  AxisMap ym, zm;
  long long pitch() const { return std::max((long long)ny * nkx, (long long)ym.nk() * ld1); }
  static constexpr const unsigned char* mask = nullptr;
  __device__ Lines in_lines(int nl) const {
    return lines_of((unsigned)ny * (unsigned)nkx, zm, false, nl);
  }
  __device__ Lines out_lines(int nl) const {
    return lines_all((unsigned)ym.nk() * (unsigned)ld1, zm.n, nl);
  }
  __device__ long long in_plane(int o) const { return (long long)ym.full(o) * nkx; }
  __device__ long long out_plane(int o) const { return (long long)o * ld1; }
};

// y-pass, inverse: W1 (nz, nyk, ld1) -> W2 (nz, ny, ld2); planes are z.
template <typename T>
struct OpYInv3 : PlainRun<T, OpYInv3<T>> {
  StridedDesc<T> d;
  const cpx<T>* in;
  cpx<T>* out;
  long long ifs, ofs;
  int ny, ld1, ld2;
  AxisMap ym;
  long long pitch() const { return ld1 > ld2 ? ld1 : ld2; }
  static constexpr const unsigned char* mask = nullptr;
  __device__ Lines in_lines(int nl) const { return lines_of(ld1, ym, true, nl); }
  __device__ Lines out_lines(int nl) const { return lines_all(ld2, ny, nl); }
  __device__ long long in_plane(int z) const { return (long long)z * ym.nk() * ld1; }
  __device__ long long out_plane(int z) const { return (long long)z * ny * ld2; }
};

// y-pass, forward: W2 (nz, ny, ld2) -> W1 (nz, nyk, ld1).
template <typename T>
struct OpYFwd3 : PlainRun<T, OpYFwd3<T>> {
  StridedDesc<T> d;
  const cpx<T>* in;
  cpx<T>* out;
  long long ifs, ofs;
  int ny, ld1, ld2;
  AxisMap ym;
  long long pitch() const { return ld1 > ld2 ? ld1 : ld2; }
  static constexpr const unsigned char* mask = nullptr;
  __device__ Lines in_lines(int nl) const { return lines_all(ld2, ny, nl); }
  __device__ Lines out_lines(int nl) const { return lines_of(ld1, ym, true, nl); }
  __device__ long long in_plane(int z) const { return (long long)z * ny * ld2; }
  __device__ long long out_plane(int z) const { return (long long)z * ym.nk() * ld1; }
};

// z-pass, forward: W1 (nz, nyk, ld1) -> K (nz, ny, nkx); only kept modes
// are written, dealiased ones (mask) as zero.
template <typename T>
struct OpZFwd : PlainRun<T, OpZFwd<T>> {
  StridedDesc<T> d;
  const cpx<T>* in;
  cpx<T>* out;
  long long ifs, ofs;
  int ny, nkx, ld1;
  AxisMap ym, zm;
  const unsigned char* mask;
  long long pitch() const { return std::max((long long)ny * nkx, (long long)ym.nk() * ld1); }
  __device__ Lines in_lines(int nl) const {
    return lines_all((unsigned)ym.nk() * (unsigned)ld1, zm.n, nl);
  }
  __device__ Lines out_lines(int nl) const {
    return lines_of((unsigned)ny * (unsigned)nkx, zm, false, nl);
  }
  __device__ long long in_plane(int o) const { return (long long)o * ld1; }
  __device__ long long out_plane(int o) const { return (long long)ym.full(o) * nkx; }
};

// 2D y-pass, inverse: K (ny, nkx) -> W2 (ny, ld2).
template <typename T>
struct OpYInv2 : PlainRun<T, OpYInv2<T>> {
  StridedDesc<T> d;
  const cpx<T>* in;
  cpx<T>* out;
  long long ifs, ofs;
  int nkx, ld2;
  AxisMap ym;
  long long pitch() const { return nkx > ld2 ? nkx : ld2; }
  static constexpr const unsigned char* mask = nullptr;
  __device__ Lines in_lines(int nl) const { return lines_of(nkx, ym, false, nl); }
  __device__ Lines out_lines(int nl) const { return lines_all(ld2, ym.n, nl); }
  __device__ long long in_plane(int) const { return 0; }
  __device__ long long out_plane(int) const { return 0; }
};

// 2D y-pass, forward: W2 (ny, ld2) -> K (ny, nkx), kept modes only.
template <typename T>
struct OpYFwd2 : PlainRun<T, OpYFwd2<T>> {
  StridedDesc<T> d;
  const cpx<T>* in;
  cpx<T>* out;
  long long ifs, ofs;
  int nkx, ld2;
  AxisMap ym;
  const unsigned char* mask;
  long long pitch() const { return nkx > ld2 ? nkx : ld2; }
  __device__ Lines in_lines(int nl) const { return lines_all(ld2, ym.n, nl); }
  __device__ Lines out_lines(int nl) const { return lines_of(nkx, ym, false, nl); }
  __device__ long long in_plane(int) const { return 0; }
  __device__ long long out_plane(int) const { return 0; }
};

// ns3d z-pass, inverse, with the curl folded in.  omega = i k x v needs
// i kz v only through d/dz, which is a transform of its own along z, while
// kx and ky are constant on a z column and multiply after the transform:
//   omega_x = i ky Vz - Dz[vy],  omega_y = Dz[vx] - i kx Vz,
//   omega_z = i kx Vy - i ky Vx (+ f on the kx = ky = 0 column),
// with V = iFFT_z(v) and Dz[a] = iFFT_z(i kz a).  Five transforms per column,
// each input read from HBM once; outputs 0-2 are v, 3-5 omega.
template <typename T>
struct OpZInvCurl {
  static constexpr bool kMulti = true;  // several transforms of a line in registers
  static constexpr bool kFieldPerBlock = false;
  StridedDesc<T> d;
  const cpx<T>* in;  // 3 fields
  cpx<T>* out;       // 6 fields
  long long ifs, ofs;
  int ny, nz, nkx, ld1;
  AxisMap ym, zm;
  T dkx, dky, dkz;
  int has_f;
  T fcor;
  int with_b;  // ns3d.strat: input 3 (b) transformed into output 6
  long long pitch() const { return std::max((long long)ny * nkx, (long long)ym.nk() * ld1); }

  template <int DIR, int LOGN, int LOGE>
  __device__ __forceinline__ void run(cpx<T>* buf, const cpx<T>* tw, int o, int line0) const {
    constexpr int E = 1 << LOGE;
    const int nl = d.nlines - line0;
    const int iy = ym.full(o);
    const T ky = T(ksigned(iy, ny)) * dky;
    const Lines gi = lines_of((unsigned)ny * (unsigned)nkx, zm, false, nl);
    const Lines go = lines_all((unsigned)ym.nk() * (unsigned)ld1, nz, nl);
    const cpx<T>* in0 = in + (long long)iy * nkx + line0;
    cpx<T>* out0 = out + (long long)o * ld1 + line0;
    cpx<T> sVz[E], sv[E], sVy[E];
    auto ld = [&](int c, const Slot& t) { return ln_load<LOGN, T>(gi, in0 + c * ifs, t); };
    auto st = [&](int c, const Slot& t, cpx<T> v) { ln_store<LOGN, T>(go, out0 + c * ofs, t, v); };
    // (not shared between its two uses: eight registers for a transform)
    auto kz_of = [&](const Slot& t) {
      int p = t.pos();
      asm volatile("" : "+v"(p));
      return T(ksigned(p, nz)) * dkz;
    };
    auto kx_of = [&](const Slot& t) { return T(line0 + t.line) * dkx; };
    // Each input is loaded once, into sv (vy, then vx) or sVz (b, once Vz
    // is no longer needed), while the transform before the one that first
    // uses it runs (tile_fft's fetch hook): only the first load of a tile
    // waits for HBM.
    // Vz; vy fetched
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL, [&](const Slot& t) { return ld(2, t); },
        [&](const Slot& t, cpx<T> v) {
          sVz[t.e] = v;
          st(2, t, v);
        },
        [&](const Slot& t) { sv[t.e] = ld(1, t); });
    // omega_x = i ky Vz - Dz[vy]
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL,
        [&](const Slot& t) { return mul_i(scale(sv[t.e], kz_of(t))); },
        [&](const Slot& t, cpx<T> v) { st(3, t, mul_i(scale(sVz[t.e], ky)) - v); });
    // Vy; vx fetched over vy once the first stage has read it
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL, [&](const Slot& t) { return sv[t.e]; },
        [&](const Slot& t, cpx<T> v) {
          sVy[t.e] = v;
          st(1, t, v);
        },
        [&](const Slot& t) { sv[t.e] = ld(0, t); });
    // omega_y = Dz[vx] - i kx Vz
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL,
        [&](const Slot& t) { return mul_i(scale(sv[t.e], kz_of(t))); },
        [&](const Slot& t, cpx<T> v) { st(4, t, v - mul_i(scale(sVz[t.e], kx_of(t)))); });
    // Vx and omega_z = i kx Vy - i ky Vx (+ f); b fetched into sVz
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL, [&](const Slot& t) { return sv[t.e]; },
        [&](const Slot& t, cpx<T> v) {
          st(0, t, v);
          cpx<T> w = mul_i(scale(sVy[t.e], kx_of(t)) - scale(v, ky));
          if (has_f && iy == 0 && line0 + t.line == 0) w.x += fcor;
          st(5, t, w);
        },
        [&](const Slot& t) {
          if (with_b) sVz[t.e] = ld(3, t);
        });
    if (with_b)
      tile_fft<T, DIR, LOGN, LOGE>(
          buf, tw, d, d.logL, [&](const Slot& t) { return sVz[t.e]; },
          [&](const Slot& t, cpx<T> v) { st(6, t, v); });
  }
};

// ns2d y-pass, inverse, from the vorticity: one read of rot, four
// transforms: ux = i ky rot / k^2, uy = -i kx rot / k^2, d_x rot = i kx rot,
// d_y rot = i ky rot (k^2 = 1e-14 at k = 0, the K2_not0 convention).
template <typename T>
struct OpYInv2NS {
  static constexpr bool kMulti = false;
  static constexpr bool kFieldPerBlock = false;
  // the four outputs can share one tile as 4 L lines (small transforms)
  static constexpr int kLineMul = 4;
  // whether the stacked outputs are in reach of a 32-bit offset
  bool stack_ok() const { return (4.0 * ofs) * sizeof(cpx<T>) < kBufMax; }
  StridedDesc<T> d;
  const cpx<T>* in;
  cpx<T>* out;
  long long ofs;
  // plane o of a batch of independent runs: in + o * ips, out + o * ops
  long long ips = 0, ops = 0;
  int ny, nkx, ld2;
  AxisMap ym;
  T dkx, dky;
  long long pitch() const { return nkx > ld2 ? nkx : ld2; }

  // multiplier (without i) of output c at (line, p); applied with
  // scale_rounded, so that the forms of the pass below give the same bits
  __device__ __forceinline__ T factor(int c, int line, int p) const {
    const T kx = T(line) * dkx, ky = T(ksigned(p, ny)) * dky;
    if (c >= 2) return c == 2 ? kx : ky;
    T k2 = fma_t(kx, kx, ky * ky);
    if (k2 == T(0)) k2 = T(1e-14);
    return (c == 0 ? ky : -kx) * (T(1) / k2);
  }

  template <int DIR, int LOGN, int LOGE>
  __device__ __forceinline__ void run(cpx<T>* buf, const cpx<T>* tw, int o, int line0) const {
    constexpr int E = 1 << LOGE;
    const int nl = d.nlines - line0;
    const Lines gi = lines_of(nkx, ym, false, nl), go = lines_all(ld2, ny, nl);
    const cpx<T>* in0 = in + o * ips + line0;
    cpx<T>* out0 = out + o * ops + line0;
    if (d.stack) {
      // one transform of 4 L lines: line l is output l >> logL of line
      // l & (L - 1), each line computed as in the sequential form below
      const int lm = (1 << d.logL) - 1;
      tile_fft<T, DIR, LOGN, LOGE>(
          buf, tw, d, d.logL + 2,
          [&](const Slot& t) {
            const Slot u{t.e, t.line & lm, t.j, t.pr};
            const cpx<T> r = ln_load<LOGN, T>(gi, in0, u);
            return mul_i(scale_rounded(r, factor(t.line >> d.logL, line0 + u.line, t.pos())));
          },
          [&](const Slot& t, cpx<T> v) {
            const Slot u{t.e, t.line & lm, t.j, t.pr};
            const int c = t.line >> d.logL;
            if constexpr (LOGN > 0) {
              // the output field is part of the lane's offset (the launcher
              // stacks only where it fits 32 bits)
              const unsigned off = ln_lane(go, u, sizeof(cpx<T>)) +
                                   (unsigned)c * (unsigned)ofs * (unsigned)sizeof(cpx<T>);
              buf_store<T>(buf_rsrc(out0 + ln_base<LOGN>(go, u), kBufMax),
                           ln_kept<LOGN>(go, u) ? off : kOOB, v);
            } else {
              ln_store<LOGN, T>(go, out0 + c * ofs, u, v);
            }
          });
      return;
    }
    cpx<T> sr[E];
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL,
        [&](const Slot& t) {
          sr[t.e] = ln_load<LOGN, T>(gi, in0, t);
          return mul_i(scale_rounded(sr[t.e], factor(0, line0 + t.line, t.pos())));
        },
        [&](const Slot& t, cpx<T> v) { ln_store<LOGN, T>(go, out0, t, v); });
#pragma unroll
    for (int c = 1; c < 4; ++c)
      tile_fft<T, DIR, LOGN, LOGE>(
          buf, tw, d, d.logL,
          [&](const Slot& t) {
            return mul_i(scale_rounded(sr[t.e], factor(c, line0 + t.line, t.pos())));
          },
          [&](const Slot& t, cpx<T> v) { ln_store<LOGN, T>(go, out0 + c * ofs, t, v); });
  }
};

// OpYInv2NS with one output field per workgroup (blockIdx.y): four times
// the workgroups, a quarter of the serial work each, the input read once per
// output (long transforms with few lines, such as ns2d at 2048^2).
template <typename T>
struct OpYInv2NSOne : OpYInv2NS<T> {
  static constexpr bool kFieldPerBlock = true;
  // the same stages as OpYInv2NS on the same problem: the same bits
  static constexpr bool kWavesPerField = true;
  static constexpr int kLineMul = 1;

  template <int DIR, int LOGN, int LOGE>
  __device__ __forceinline__ void run(cpx<T>* buf, const cpx<T>* tw, int o, int line0) const {
    const StridedDesc<T>& d = this->d;
    const int nl = d.nlines - line0;
    const int c = blockIdx.y;
    const Lines gi = lines_of(this->nkx, this->ym, false, nl);
    const Lines go = lines_all(this->ld2, this->ny, nl);
    const cpx<T>* in0 = this->in + o * this->ips + line0;
    cpx<T>* out0 = this->out + o * this->ops + c * this->ofs + line0;
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL,
        [&](const Slot& t) {
          const cpx<T> r = ln_load<LOGN, T>(gi, in0, t);
          return mul_i(scale_rounded(r, this->factor(c, line0 + t.line, t.pos())));
        },
        [&](const Slot& t, cpx<T> v) { ln_store<LOGN, T>(go, out0, t, v); });
  }
};

// The pass's own argument struct through the kernel-argument pointer, which
// the optimizer cannot follow back: what is read through it is loaded where
// it is used, after the transforms, instead of being held in (and spilled
// from) scalar registers from the start of the kernel.
template <class Op>
__device__ __forceinline__ const Op& late_args() {
  auto* p = __builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const Op*)(const void*)p;
}

// Runge-Kutta stage of the modes in a tile's output slots: N(e, n) gives the
// NV tendencies of slot e (masked here).  The state streams of two
// slots are loaded before any is used, so that their latencies overlap.
template <typename T, int NV>
constexpr int rk_batch() {
  return NV > 3 ? 1 : 2;
}
template <typename T, int NV, int LOGN, int LOGE, class NFn>
__device__ __forceinline__ void rk_slots(const StridedDesc<T>& d, const Lines& g,
                                         const RKArgs<T>& rk, const Visc& visc, double dt,
                                         const unsigned char* mask, long long base, int line0,
                                         bool along_z, int iky, const NFn& tend) {
  constexpr int E = 1 << LOGE;
  constexpr int B = rk_batch<T, NV>();
#pragma unroll
  for (int e0 = 0; e0 < E; e0 += B) {
    std::conditional_t<B == 1, RKDirect<T>, RKStreams<T, NV>> st[B];
#pragma unroll
    for (int q = 0; q < B; ++q) {
      Slot t;
      if (!last_slot<LOGN, LOGE>(e0 + q, d, d.logL, t)) continue;
      rk_load(rk, SlotMode<LOGN, T>{g, t, base}, st[q]);
    }
#pragma unroll
    for (int q = 0; q < B; ++q) {
      Slot t;
      if (!last_slot<LOGN, LOGE>(e0 + q, d, d.logL, t)) continue;
      if (B == 1) {
        // nothing of one slot is kept in registers for the next
        asm volatile("" : "+v"(t.j), "+v"(t.line));
      }
      if (!ln_kept<LOGN>(g, t)) continue;
      const SlotMode<LOGN, T> m{g, t, base};
      cpx<T> N[NV];
      tend(t, m, N);
      if (ln_masked<LOGN>(g, mask, t)) {
#pragma unroll
        for (int v = 0; v < NV; ++v) N[v] = zero<T>();
      }
      const int kp = ksigned(t.pos(), d.N);
      rk_point<T, NV>(rk, visc, dt, m, line0 + t.line, along_z ? iky : kp, along_z ? kp : 0, st[q],
                      N);
    }
  }
}

// ns3d z-pass, forward, with the Runge-Kutta stage folded in: the three
// tendency components are transformed one after the other (the first two
// kept in registers), then each kept mode is projected, masked and advanced
// (rk_point); the tendency never goes to HBM.
template <typename T>
struct OpZFwdRK3 {
  static constexpr bool kMulti = true;
  static constexpr bool kFieldPerBlock = false;
  StridedDesc<T> d;
  const cpx<T>* in;  // W1, 3 fields
  long long ifs;
  int ny, nkx, ld1;
  AxisMap ym, zm;
  const unsigned char* mask;
  RKArgs<T> rk;
  long long pitch() const { return std::max((long long)ny * nkx, (long long)ym.nk() * ld1); }

  template <int DIR, int LOGN, int LOGE>
  __device__ __forceinline__ void run(cpx<T>* buf, const cpx<T>* tw, int o, int line0) const {
    constexpr int E = 1 << LOGE;
    const int nl = d.nlines - line0;
    const int iy = ym.full(o);
    const Lines gi = lines_all((unsigned)ym.nk() * (unsigned)ld1, d.N, nl);
    const Lines gk = lines_of((unsigned)ny * (unsigned)nkx, zm, false, nl);
    const cpx<T>* in0 = in + (long long)o * ld1 + line0;
    const long long base = (long long)iy * nkx + line0;
    cpx<T> s0[E], s1[E], s2[E];
    auto ld = [&](int c, const Slot& t) { return ln_load<LOGN, T>(gi, in0 + c * ifs, t); };
    // input c + 1 is fetched into s(c+1) while transform c runs; the
    // stash's first stage reads it before its last stage stores the output
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL, [&](const Slot& t) { return ld(0, t); },
        [&](const Slot& t, cpx<T> v) { s0[t.e] = v; },
        [&](const Slot& t) { s1[t.e] = ld(1, t); });
    pin(s0);
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL, [&](const Slot& t) { return s1[t.e]; },
        [&](const Slot& t, cpx<T> v) { s1[t.e] = v; },
        [&](const Slot& t) { s2[t.e] = ld(2, t); });
    pin(s1);
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL, [&](const Slot& t) { return s2[t.e]; },
        [&](const Slot& t, cpx<T> v) { s2[t.e] = v; });
    pin(s2);
    const RKArgs<T>& rk = late_args<OpZFwdRK3>().rk;
    rk_slots<T, 3, LOGN, LOGE>(d, gk, rk, rk.visc, *rk.dt, mask ? mask + base : nullptr, base,
                               line0, true, ksigned(iy, ny),
                               [&](const Slot& t, const SlotMode<LOGN, T>&, cpx<T>* N) {
                                 N[0] = s0[t.e];
                                 N[1] = s1[t.e];
                                 N[2] = s2[t.e];
                               });
  }
};

// ns3d.strat z-pass, forward, with the Runge-Kutta stage folded in
// (fluidsim/solvers/ns3d/strat/solver.py:29-33, 138-216): W1 fields 0-2 are
// the transforms of v x omega, 3-5 those of v b.  Per kept mode
//   N_v = (F_x, F_y, F_z + b),  N_b = -i k.(v b)^ - N^2 v_z,
// with b and v_z of the state the tendency is evaluated on (rk.src); the
// projection acts on N_v only (rk_point).
template <typename T>
struct OpZFwdRKStrat {
  static constexpr bool kMulti = true;
  static constexpr bool kFieldPerBlock = false;
  StridedDesc<T> d;
  const cpx<T>* in;  // W1, 6 fields
  long long ifs;
  int ny, nkx, ld1;
  AxisMap ym, zm;
  const unsigned char* mask;
  T dkx, dky, dkz;
  T N2;
  RKArgs<T> rk;
  long long pitch() const { return std::max((long long)ny * nkx, (long long)ym.nk() * ld1); }

  template <int DIR, int LOGN, int LOGE>
  __device__ __forceinline__ void run(cpx<T>* buf, const cpx<T>* tw, int o, int line0) const {
    constexpr int E = 1 << LOGE;
    const int nl = d.nlines - line0;
    const int iy = ym.full(o);
    const int iky = ksigned(iy, ny);
    const T ky = T(iky) * dky;
    const Lines gi = lines_all((unsigned)ym.nk() * (unsigned)ld1, d.N, nl);
    const Lines gk = lines_of((unsigned)ny * (unsigned)nkx, zm, false, nl);
    const cpx<T>* in0 = in + (long long)o * ld1 + line0;
    const long long base = (long long)iy * nkx + line0;
    cpx<T> s0[E], s1[E], s2[E], sb[E];
    auto ld = [&](int c, const Slot& t) { return ln_load<LOGN, T>(gi, in0 + c * ifs, t); };
    // The v b transforms first: their sum sb is one register array, where
    // the three tendencies would all be live during them (with the sum last
    // the pass needs more than 128 registers).  Each input is fetched while
    // the transform before runs (see OpZFwdRK3).
    // sb = kx G_x + ky G_y + kz G_z  (N_b = -i sb - N^2 v_z)
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL, [&](const Slot& t) { return ld(3, t); },
        [&](const Slot& t, cpx<T> v) { sb[t.e] = scale(v, T(line0 + t.line) * dkx); },
        [&](const Slot& t) { s0[t.e] = ld(4, t); });
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL, [&](const Slot& t) { return s0[t.e]; },
        [&](const Slot& t, cpx<T> v) { sb[t.e] = sb[t.e] + scale(v, ky); },
        [&](const Slot& t) { s1[t.e] = ld(5, t); });
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL, [&](const Slot& t) { return s1[t.e]; },
        [&](const Slot& t, cpx<T> v) {
          sb[t.e] = sb[t.e] + scale(v, T(ksigned(t.pos(), d.N)) * dkz);
        },
        [&](const Slot& t) { s0[t.e] = ld(0, t); });
    pin(sb);
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL, [&](const Slot& t) { return s0[t.e]; },
        [&](const Slot& t, cpx<T> v) { s0[t.e] = v; },
        [&](const Slot& t) { s1[t.e] = ld(1, t); });
    pin(s0);
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL, [&](const Slot& t) { return s1[t.e]; },
        [&](const Slot& t, cpx<T> v) { s1[t.e] = v; },
        [&](const Slot& t) { s2[t.e] = ld(2, t); });
    pin(s1);
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL, [&](const Slot& t) { return s2[t.e]; },
        [&](const Slot& t, cpx<T> v) { s2[t.e] = v; });
    pin(s2);
    const RKArgs<T>& rk = late_args<OpZFwdRKStrat>().rk;
    rk_slots<T, 4, LOGN, LOGE>(
        d, gk, rk, rk.visc, *rk.dt, mask ? mask + base : nullptr, base, line0, true, iky,
        [&](const Slot& t, const SlotMode<LOGN, T>& m, cpx<T>* N) {
          const cpx<T> bs = m.load(rk.src[3]), vzs = m.load(rk.src[2]);
          N[0] = s0[t.e];
          N[1] = s1[t.e];
          N[2] = s2[t.e] + bs;
          N[3] = scale(mul_i(sb[t.e]), T(-1)) - scale(vzs, N2);
        });
  }
};

// ns2d y-pass, forward, with the Runge-Kutta stage folded in.
template <typename T>
struct OpYFwd2RK {
  static constexpr bool kMulti = false;
  static constexpr bool kFieldPerBlock = false;
  StridedDesc<T> d;
  const cpx<T>* in;  // W2, 1 field
  int ny, nkx, ld2;
  AxisMap ym;
  const unsigned char* mask;
  RKArgs<T> rk;
  // plane o of a batch of independent runs: W2 rows at o * ips, state modes
  // at o * ops, and the run's dt and viscosities at bpar[5 o .. 5 o + 4]
  // (dt, nu_2, nu_4, nu_8, nu_m4); bpar null: rk.dt and rk.visc
  long long ips = 0, ops = 0;
  const double* bpar = nullptr;
  long long pitch() const { return nkx > ld2 ? nkx : ld2; }

  template <int DIR, int LOGN, int LOGE>
  __device__ __forceinline__ void run(cpx<T>* buf, const cpx<T>* tw, int o, int line0) const {
    constexpr int E = 1 << LOGE;
    const int nl = d.nlines - line0;
    const cpx<T>* in0 = in + o * ips + line0;
    const Lines gi = lines_all(ld2, ny, nl), gk = lines_of(nkx, ym, false, nl);
    double dt;
    Visc visc;
    if (bpar) {
      const double* q = bpar + 5 * o;
      dt = q[0];
      visc = Visc{q[1], q[2], q[3], q[4]};
    } else {
      dt = *rk.dt;
      visc = rk.visc;
    }
    cpx<T> s0[E];
    tile_fft<T, DIR, LOGN, LOGE>(
        buf, tw, d, d.logL, [&](const Slot& t) { return ln_load<LOGN, T>(gi, in0, t); },
        [&](const Slot& t, cpx<T> v) { s0[t.e] = v; });
    pin(s0);
    rk_slots<T, 1, LOGN, LOGE>(
        d, gk, rk, visc, dt, mask ? mask + line0 : nullptr, o * ops + line0, line0, false, 0,
        [&](const Slot& t, const SlotMode<LOGN, T>&, cpx<T>* N) { N[0] = s0[t.e]; });
  }
};

// ---------------------------------------------------------------- rows
template <typename T>
struct XDesc {
  // M complex points per row: nx / 2, odd nx nx; RB rows per workgroup.  The
  // logarithms are -1 in k_xpass_gen, where M and RB are any numbers
  int nx, lognx, M, logM;
  int RB, logRB;
  int nrows;
  int nf_in, nf_out;
  int mx_in, ld_in;    // kept kx and row stride of the c2r input rows
  int mx_out, ld_out;  // kept kx and row stride of the r2c output rows
  long long ifs, ofs;  // field strides (elements)
  T scale;             // applied to the r2c output
  const cpx<T>* tw;    // exp(-2 pi i m / nx), m < nx (copied to LDS)
  // mixed-radix stages of a length-M complex transform (k_xpass_gen)
  int nst, inplace;
  int rad[kMaxStages];
};

template <typename T>
__device__ __forceinline__ T wave_max(T v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  return v;
}

// Block-wide max of up to 3 values, then one atomicMax per value on the bit
// pattern of a non-negative double (monotonic as unsigned 64-bit).
template <typename T, int kT>
__device__ void block_max_atomic(T m0, T m1, T m2, int nv,
                                 unsigned long long* dst) {
  __shared__ T red[3][kT / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  m0 = wave_max(m0);
  m1 = wave_max(m1);
  m2 = wave_max(m2);
  if (lane == 0) {
    red[0][wid] = m0;
    red[1][wid] = m1;
    red[2][wid] = m2;
  }
  __syncthreads();
  if (threadIdx.x < nv) {
    T m = red[threadIdx.x][0];
    for (int w = 1; w < kT / 64; ++w) m = fmax(m, red[threadIdx.x][w]);
    const double md = (double)m;
    atomicMax(dst + threadIdx.x, (unsigned long long)__double_as_longlong(md));
  }
  __syncthreads();
}

// Real view of the padded row layout: real x of line lr.
__device__ __forceinline__ int rpad(int lr, int x, int ldr) {
  return 2 * (lr * ldr + lpad(x >> 1)) + (x & 1);
}

// At least 4 waves per SIMD (caps the VGPR count).
template <typename T, int EPT, int kT, class Op>
static __global__ __launch_bounds__(kT) __attribute__((amdgpu_waves_per_eu(4)))
void k_xpass(Op op) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const XDesc<T>& d = op.d;
  cpx<T>* s_tw = reinterpret_cast<cpx<T>*>(smem_raw);
  cpx<T>* buf = s_tw + d.nx;
  T* bufr = reinterpret_cast<T*>(buf);
  const int M = d.M, logM = d.logM, nx = d.nx;
  const int H = M >> 1, logH = logM - 1;
  const int ldr = lpad(M);  // padded complex row stride in LDS
  const int row0 = blockIdx.x << d.logRB;
  const int tid = threadIdx.x;
  for (int i = tid; i < nx; i += kT) s_tw[i] = d.tw[i];
  __syncthreads();

  if constexpr (Op::kInv) {
    // c2r pre-processing, one thread per pair (k, M - k):
    // Z[k] = (X[k] + conj X[M-k]) + i conj(W^k) (X[k] - conj X[M-k]),
    // W = exp(-2 pi i / nx); only the real parts of X[0] and X[M] are used;
    // the k = 0 thread also does the self-paired k = M/2.  The loads of
    // kU consecutive pairs of a thread are issued before any is used, so
    // their latencies overlap.
    constexpr int kU = 4;
    const int n_in = (d.nf_in << d.logRB) << logH;
    for (int base = tid; base < n_in; base += kU * kT) {
      cpx<T> Xk[kU], Xm[kU], Xh[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int idx = base + u * kT;
        Xk[u] = zero<T>();
        Xm[u] = zero<T>();
        Xh[u] = zero<T>();
        const int k = idx & (H - 1);
        const int lr = idx >> logH;
        const int row = row0 + (lr & (d.RB - 1));
        if (idx < n_in && row < d.nrows) {
          const cpx<T>* src = op.in + (lr >> d.logRB) * d.ifs + (long long)row * d.ld_in;
          if (k < d.mx_in) Xk[u] = src[k];
          if (M - k < d.mx_in) Xm[u] = src[M - k];
          if (k == 0 && H < d.mx_in) Xh[u] = src[H];
        }
      }
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int idx = base + u * kT;
        if (idx >= n_in) break;
        const int k = idx & (H - 1);
        const int lr = idx >> logH;
        cpx<T>* Z = buf + lr * ldr;
        if (k == 0) {
          Xk[u].y = T(0);
          Xm[u].y = T(0);
        }
        const cpx<T> w = s_tw[k];
        const cpx<T> dk = Xk[u] - conj(Xm[u]), dm = Xm[u] - conj(Xk[u]);
        Z[lpad(k)] = (Xk[u] + conj(Xm[u])) + mul_i(conj(w) * dk);
        if (k == 0) {
          const cpx<T> dh = Xh[u] - conj(Xh[u]);
          Z[lpad(H)] = (Xh[u] + conj(Xh[u])) + mul_i(conj(s_tw[H]) * dh);
        } else {
          // conj(W^(M-k)) = -W^k
          Z[lpad(M - k)] = (Xm[u] + conj(Xk[u])) - mul_i(w * dm);
        }
      }
    }
    __syncthreads();
    lds_fft_rows<T, +1, EPT, kT>(buf, logM, d.nf_in << d.logRB, ldr, s_tw, 1);
  } else {
    const int n_in = (d.nf_in << d.logRB) << d.lognx;
    for (int idx = tid; idx < n_in; idx += kT) {
      const int x = idx & (nx - 1);
      const int lr = idx >> d.lognx;
      const int f = lr >> d.logRB;
      const int row = row0 + (lr & (d.RB - 1));
      bufr[rpad(lr, x, ldr)] =
          row < d.nrows ? op.inr[f * d.ifs + (long long)row * nx + x] : T(0);
    }
    __syncthreads();
  }

  if constexpr (Op::kStoreReal) {
    const int n_out = (d.nf_in << d.logRB) << d.lognx;
    for (int idx = tid; idx < n_out; idx += kT) {
      const int x = idx & (nx - 1);
      const int lr = idx >> d.lognx;
      const int f = lr >> d.logRB;
      const int row = row0 + (lr & (d.RB - 1));
      if (row < d.nrows) op.outr[f * d.ofs + (long long)row * nx + x] = bufr[rpad(lr, x, ldr)];
    }
    return;
  } else {
    op.physical(bufr, row0, ldr);
    __syncthreads();
    lds_fft_rows<T, -1, EPT, kT>(buf, logM, d.nf_out << d.logRB, ldr, s_tw, 1);
    // r2c post-processing, one thread per pair (k, M - k):
    // E = (Z[k] + conj Z[M-k]) / 2, O = -i (Z[k] - conj Z[M-k]) / 2,
    // X[k] = E + W^k O, X[M-k] = conj(E - W^k O); k = 0 also does M/2.
    const int n_out = (d.nf_out << d.logRB) << logH;
    for (int idx = tid; idx < n_out; idx += kT) {
      const int k = idx & (H - 1);
      const int lr = idx >> logH;
      const int f = lr >> d.logRB;
      const int row = row0 + (lr & (d.RB - 1));
      if (row >= d.nrows) continue;
      const cpx<T>* Z = buf + lr * ldr;
      cpx<T>* dst = op.out + f * d.ofs + (long long)row * d.ld_out;
      const T h = T(0.5);
      {
        const cpx<T> Zk = Z[lpad(k)], Zm = conj(Z[lpad((M - k) & (M - 1))]);
        const cpx<T> E = scale(Zk + Zm, h), dd = Zk - Zm;
        const cpx<T> P = s_tw[k] * mk<T>(dd.y * h, -dd.x * h);
        if (k < d.mx_out) dst[k] = scale(E + P, d.scale);
        if (M - k < d.mx_out) dst[M - k] = scale(conj(E - P), d.scale);
      }
      if (k == 0 && H < d.mx_out) {
        const cpx<T> Zk = Z[lpad(H)], Zm = conj(Z[lpad(H)]);
        const cpx<T> E = scale(Zk + Zm, h), dd = Zk - Zm;
        const cpx<T> P = s_tw[H] * mk<T>(dd.y * h, -dd.x * h);
        dst[H] = scale(E + P, d.scale);
      }
    }
  }
}

// Row pass of any length nx (grids that are not powers of two).  Even nx:
// a real row is one complex transform of length M = nx/2, z[j] = x[2j] +
// i x[2j+1], with the pairing of k and M - k before and after it as in
// k_xpass (computed per element, both operands read from memory, the second
// from cache).  Odd nx: one complex transform of length M = nx of the half
// spectrum extended by Hermitian symmetry, whose real part is the row (the
// imaginary part of X[0] drops out, as in numpy's irfft).  The products run
// per point (Op::point).  Rows per workgroup: d.RB (any count), fields
// stacked as rows f RB + r of stride M in one or two LDS buffers (gen_fft).
template <typename T, class Op>
static __global__ __launch_bounds__(kGenThr, 4) void k_xpass_gen(Op op) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int kT = kGenThr;
  const XDesc<T>& d = op.d;
  const int nx = d.nx, RB = d.RB, M = d.M;
  const bool half = M != nx;
  cpx<T>* s_tw = reinterpret_cast<cpx<T>*>(smem_raw);
  const int nfm = d.nf_in > d.nf_out ? d.nf_in : d.nf_out;
  cpx<T>* A = s_tw + nx;
  cpx<T>* B = d.inplace ? A : A + nfm * RB * M;
  const int row0 = blockIdx.x * RB;
  const int tid = threadIdx.x;
  const TileLayout lay{M, 1};
  const unsigned mM = magic_of(M), mRB = magic_of(RB);
  for (int i = tid; i < nx; i += kT) s_tw[i] = d.tw[i];
  __syncthreads();
  const int n_in = d.nf_in * RB * M;
  // the loads of kU elements of a thread are issued before any is used; what
  // is masked (dealiased modes, rows past the end) reads element 0 instead
  constexpr int kU = 4;
  for (int base = tid; base < n_in; base += kU * kT) {
    cpx<T> Xk[kU], Xm[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int idx = base + u * kT < n_in ? base + u * kT : 0;
      const int lr = magic_div(idx, mM, M), x = idx - lr * M;
      const int f = magic_div(lr, mRB, RB), row = row0 + (lr - f * RB);
      const bool in = row < d.nrows;
      if constexpr (Op::kInv) {
        const cpx<T>* src = op.in + (in ? f * d.ifs + (long long)row * d.ld_in : 0);
        const int k = half || x <= nx / 2 ? x : nx - x;
        const bool okk = in && k < d.mx_in, okm = in && half && M - x < d.mx_in;
        Xk[u] = src[okk ? k : 0];
        Xm[u] = src[okm ? M - x : 0];
        if (!okk) Xk[u] = zero<T>();
        if (!okm) Xm[u] = zero<T>();
      } else {
        const T* src = op.inr + (in ? f * d.ifs + (long long)row * nx : 0);
        Xk[u] = half ? mk<T>(src[2 * x], src[2 * x + 1]) : mk<T>(src[x], T(0));
        if (!in) Xk[u] = zero<T>();
      }
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int idx = base + u * kT;
      if (idx >= n_in) break;
      const int x = idx - magic_div(idx, mM, M) * M;
      cpx<T> v = Xk[u];
      if constexpr (Op::kInv) {
        if (half) {
          if (x == 0) Xk[u].y = Xm[u].y = T(0);
          const cpx<T> w = s_tw[x];
          const cpx<T> dk = Xk[u] - conj(Xm[u]);
          v = (Xk[u] + conj(Xm[u])) + mul_i(conj(w) * dk);
        } else if (x > nx / 2) {
          v = conj(v);
        }
      }
      A[idx] = v;
    }
  }
  __syncthreads();
  cpx<T>* res = A;
  if constexpr (Op::kInv) {
    res = gen_fft<T, +1, kT>(A, B, lay, s_tw, half ? 2 : 1, M, d.nf_in * RB, -1, d.nst, d.rad);
    if constexpr (Op::kStoreReal) {
      for (int idx = tid; idx < n_in; idx += kT) {
        const int lr = magic_div(idx, mM, M), x = idx - lr * M;
        const int f = magic_div(lr, mRB, RB), row = row0 + (lr - f * RB);
        if (row >= d.nrows) continue;
        T* dst = op.outr + f * d.ofs + (long long)row * nx;
        const cpx<T> v = res[idx];
        if (half) {
          dst[2 * x] = v.x;
          dst[2 * x + 1] = v.y;
        } else {
          dst[x] = v.x;
        }
      }
      return;
    } else {
      T m[3] = {0, 0, 0};
      const int fs = RB * M;  // elements per field
      for (int idx = tid; idx < fs; idx += kT) {
        const int r = magic_div(idx, mM, M);
        T v[8], u[8];
        for (int c = 0; c < d.nf_in && c < 8; ++c) {
          const cpx<T> z = res[c * fs + idx];
          v[c] = z.x;
          u[c] = z.y;
        }
        T mm[3] = {0, 0, 0};
        op.point(v, mm);
        if (half) op.point(u, mm);
        if (row0 + r < d.nrows)
          for (int c = 0; c < 3; ++c) m[c] = fmax(m[c], mm[c]);
        for (int c = 0; c < d.nf_out; ++c) res[c * fs + idx] = mk<T>(v[c], half ? u[c] : T(0));
      }
      if constexpr (Op::kNMax > 0)
        if (op.maxima) block_max_atomic<T, kT>(m[0], m[1], m[2], Op::kNMax, op.maxima);
      __syncthreads();
    }
  }
  cpx<T>* other = d.inplace ? res : (res == A ? B : A);
  res = gen_fft<T, -1, kT>(res, other, lay, s_tw, half ? 2 : 1, M, d.nf_out * RB, -1, d.nst,
                           d.rad);
  const int n_out = d.nf_out * RB * d.mx_out;
  const unsigned mx = magic_of(d.mx_out);
  for (int idx = tid; idx < n_out; idx += kT) {
    const int lr = magic_div(idx, mx, d.mx_out), k = idx - lr * d.mx_out;
    const int f = magic_div(lr, mRB, RB), row = row0 + (lr - f * RB);
    if (row >= d.nrows) continue;
    const cpx<T>* Z = res + lr * M;
    cpx<T> X = Z[k < M ? k : 0];  // Z[M] = Z[0]
    if (half) {
      // X[k] = (Zk + conj Z[M-k]) / 2 + W^k (Zk - conj Z[M-k]) / (2 i)
      const cpx<T> Zm = conj(Z[k == 0 || k == M ? 0 : M - k]);
      const cpx<T> w = k == M ? mk<T>(T(-1), T(0)) : s_tw[k];
      const cpx<T> dd = X - Zm;
      X = scale((X + Zm) + w * mk<T>(dd.y, -dd.x), T(0.5));
    }
    op.out[f * d.ofs + (long long)row * d.ld_out + k] = scale(X, d.scale);
  }
}

// plain c2r rows: W2 rows -> X rows
template <typename T>
struct OpXC2R {
  static constexpr bool kInv = true, kStoreReal = true;
  static constexpr int kNMax = 0;
  unsigned long long* maxima = nullptr;
  __device__ void point(T*, T*) const {}
  XDesc<T> d;
  const cpx<T>* in;
  const T* inr;
  T* outr;
  cpx<T>* out;
  __device__ void physical(T*, int, int) const {}
};

// plain r2c rows: X rows -> W2 rows, scaled by 1/(number of points)
template <typename T>
struct OpXR2C {
  static constexpr bool kInv = false, kStoreReal = false;
  static constexpr int kNMax = 0;
  unsigned long long* maxima = nullptr;
  __device__ void point(T*, T*) const {}
  XDesc<T> d;
  const cpx<T>* in;
  const T* inr;
  T* outr;
  cpx<T>* out;
  __device__ void physical(T*, int, int) const {}
};

// ns3d rows: (v, omega) -> v x omega, optional CFL maxima of |v_i|.
template <typename T, int kT>
struct OpXNS3D {
  static constexpr bool kInv = true, kStoreReal = false;
  XDesc<T> d;
  const cpx<T>* in;
  const T* inr;
  T* outr;
  cpx<T>* out;
  unsigned long long* maxima;  // 3 slots or null
  static constexpr int kNMax = 3;
  // one point: v = (v, omega) -> v x omega, maxima of |v_i| into m
  __device__ void point(T* v, T* m) const {
    const T vx = v[0], vy = v[1], vz = v[2];
    v[0] = vy * v[5] - vz * v[4];
    v[1] = vz * v[3] - vx * v[5];
    v[2] = vx * v[4] - vy * v[3];
    m[0] = fmax(m[0], fabs(vx));
    m[1] = fmax(m[1], fabs(vy));
    m[2] = fmax(m[2], fabs(vz));
  }
  __device__ void physical(T* b, int row0, int ldr) const {
    const int n = d.RB << d.lognx;
    const int s = 2 * ldr * d.RB;  // reals per field
    T m0 = 0, m1 = 0, m2 = 0;
    for (int idx = threadIdx.x; idx < n; idx += kT) {
      T* p = b + rpad(idx >> d.lognx, idx & (d.nx - 1), ldr);
      const T vx = p[0], vy = p[s], vz = p[2 * s];
      const T wx = p[3 * s], wy = p[4 * s], wz = p[5 * s];
      p[0] = vy * wz - vz * wy;
      p[s] = vz * wx - vx * wz;
      p[2 * s] = vx * wy - vy * wx;
      if (row0 + (idx >> d.lognx) < d.nrows) {
        m0 = fmax(m0, fabs(vx));
        m1 = fmax(m1, fabs(vy));
        m2 = fmax(m2, fabs(vz));
      }
    }
    if (maxima) block_max_atomic<T, kT>(m0, m1, m2, 3, maxima);
  }
};

// ns3d.strat rows: (v, omega, b) -> (v x omega, v b), CFL maxima of |v_i|.
template <typename T, int kT>
struct OpXStrat {
  static constexpr bool kInv = true, kStoreReal = false;
  XDesc<T> d;
  const cpx<T>* in;
  const T* inr;
  T* outr;
  cpx<T>* out;
  unsigned long long* maxima;  // 3 slots or null
  static constexpr int kNMax = 3;
  // one point: (v, omega, b) -> (v x omega, v b), maxima of |v_i| into m
  __device__ void point(T* v, T* m) const {
    const T vx = v[0], vy = v[1], vz = v[2], bb = v[6];
    v[0] = vy * v[5] - vz * v[4];
    v[1] = vz * v[3] - vx * v[5];
    v[2] = vx * v[4] - vy * v[3];
    v[3] = vx * bb;
    v[4] = vy * bb;
    v[5] = vz * bb;
    m[0] = fmax(m[0], fabs(vx));
    m[1] = fmax(m[1], fabs(vy));
    m[2] = fmax(m[2], fabs(vz));
  }
  __device__ void physical(T* b, int row0, int ldr) const {
    const int n = d.RB << d.lognx;
    const int s = 2 * ldr * d.RB;
    T m0 = 0, m1 = 0, m2 = 0;
    for (int idx = threadIdx.x; idx < n; idx += kT) {
      T* p = b + rpad(idx >> d.lognx, idx & (d.nx - 1), ldr);
      const T vx = p[0], vy = p[s], vz = p[2 * s];
      const T wx = p[3 * s], wy = p[4 * s], wz = p[5 * s], bb = p[6 * s];
      p[0] = vy * wz - vz * wy;
      p[s] = vz * wx - vx * wz;
      p[2 * s] = vx * wy - vy * wx;
      p[3 * s] = vx * bb;
      p[4 * s] = vy * bb;
      p[5 * s] = vz * bb;
      if (row0 + (idx >> d.lognx) < d.nrows) {
        m0 = fmax(m0, fabs(vx));
        m1 = fmax(m1, fabs(vy));
        m2 = fmax(m2, fabs(vz));
      }
    }
    if (maxima) block_max_atomic<T, kT>(m0, m1, m2, 3, maxima);
  }
};

// ns2d rows: (ux, uy, d_x rot, d_y rot) -> -ux d_x rot - uy (d_y rot + beta)
template <typename T, int kT>
struct OpXNS2D {
  static constexpr bool kInv = true, kStoreReal = false;
  XDesc<T> d;
  const cpx<T>* in;
  const T* inr;
  T* outr;
  cpx<T>* out;
  unsigned long long* maxima;  // 2 slots or null
  T beta;
  static constexpr int kNMax = 2;
  // one point: (ux, uy, d_x rot, d_y rot) -> -ux d_x rot - uy (d_y rot + beta)
  __device__ void point(T* v, T* m) const {
    const T ux = v[0], uy = v[1], px = v[2], py = v[3];
    v[0] = beta == T(0) ? -ux * px - uy * py : -ux * px - uy * (py + beta);
    m[0] = fmax(m[0], fabs(ux));
    m[1] = fmax(m[1], fabs(uy));
  }
  __device__ void physical(T* b, int row0, int ldr) const {
    const int n = d.RB << d.lognx;
    const int s = 2 * ldr * d.RB;
    T m0 = 0, m1 = 0;
    for (int idx = threadIdx.x; idx < n; idx += kT) {
      T* p = b + rpad(idx >> d.lognx, idx & (d.nx - 1), ldr);
      const T ux = p[0], uy = p[s], px = p[2 * s], py = p[3 * s];
      p[0] = beta == T(0) ? -ux * px - uy * py : -ux * px - uy * (py + beta);
      if (row0 + (idx >> d.lognx) < d.nrows) {
        m0 = fmax(m0, fabs(ux));
        m1 = fmax(m1, fabs(uy));
      }
    }
    if (maxima) block_max_atomic<T, kT>(m0, m1, T(0), 2, maxima);
  }
};

}  // namespace fsx

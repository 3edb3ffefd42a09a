// Tile transforms of the strided (y and z) passes.
//
// A tile is 2^logL adjacent lines (consecutive kx, the contiguous index) of
// one axis of length N.  Power-of-two lengths run tile_fft_p2, whose length is
// a template argument: the positions a thread touches are then j + constant,
// so an element costs no index arithmetic beyond one comparison (the kept
// range of pruned axes) and one LDS address addition.  A version that took
// length and lines as run-time values spent two thirds of its vector
// instructions on addresses and branches (512^3 FP32 y-inverse: 1243 of them
// per wave for 450 of arithmetic, issued 67 % of the time; now about 600).
// What that gives depends on what else bounds a pass: the y-passes of 512^3
// were at the rate of a copy already (y-inverse 814 -> 780 us, 4.6 TB/s), the
// z-passes with the curl and with the Runge-Kutta stage go from 530 to 508 and
// from 721 to 671 us, the y-inverse of 256 runs of 128^2 from 35 to 18 us.
//
// Axes of at most 8 (FP64, several transforms of a line) or 16 points are one
// stage: each thread transforms a line in registers, without LDS.  A
// Runge-Kutta step of ns3d on 256 x 256 x 8: 187 us in FP64 and 170 in FP32
// (629 and 533 with these axes in the mixed-radix stages, 265 and 225 with
// run-time lengths), on 128 x 128 x 4: 100 and 97 us (749, 647; 174, 154).
//
// Other lengths run gen_fft (mixed radix), in one LDS buffer where the
// butterflies of all threads fit their registers, else in two.
#pragma once

#include "fsx_fft.h"

namespace fsx {

// Buffer-resource loads and stores of one complex value.  A raw buffer
// access whose byte offset is at or beyond the resource's size reads zero
// and writes nothing, so masked elements (dealiased modes, rows past the
// end) take the offset kOOB instead of a branch.
constexpr unsigned kOOB = 0xffe00000u;
// Size given to resources whose extent is not known (lane_reach: every offset
// is below it).  4 MiB short of 32 bits: the lanes of a pass over a field of
// fewer than 2^31 values, the most the element indices reach, stay 8 MiB short.
constexpr unsigned kBufMax = 0xffc00000u;
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* base,
                                                          unsigned bytes) {
  // word 3 = 0x00020000: raw (untyped) 32-bit data format on gfx9 parts
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0,
                                           (int)bytes, 0x00020000);
}
template <typename T>
__device__ __forceinline__ cpx<T> buf_load(__amdgpu_buffer_rsrc_t r, unsigned off) {
  if constexpr (sizeof(T) == 4)
    return __builtin_bit_cast(cpx<T>, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
  else
    return __builtin_bit_cast(cpx<T>, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
template <typename T>
__device__ __forceinline__ void buf_store(__amdgpu_buffer_rsrc_t r, unsigned off,
                                          cpx<T> v) {
  if constexpr (sizeof(T) == 4)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2_t, v), r, off, 0, 0);
  else
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), r, off, 0, 0);
}

constexpr int kGenThr = 256;  // threads of the mixed-radix tiles

// Largest tile of a workgroup: 64 KiB (8192 FP32 or 4096 FP64 values).
template <typename T>
constexpr int strided_tile() {
  return sizeof(T) == 4 ? 8192 : 4096;
}
// log2 of the elements per thread of the strided passes: 16 (FP32 passes of
// one transform per line) or 8 (FP64; passes that keep several transforms of
// a line in registers).
template <typename T, class Op>
constexpr int strided_loge() {
  return sizeof(T) == 4 && !Op::kMulti ? 4 : 3;
}
// Threads of a workgroup of a length-2^logn pass with 2^loge elements per
// thread, at most: a full tile's, half of it for the passes that keep several
// transforms in registers up to length 256, whose 128-byte runs need no more
// (512 threads: 256 registers each); where a thread has fewer elements than
// strided_loge (small problems, short axes), 1024 threads (four stacked lines
// of 1024), 256 for several transforms.
template <typename T, class Op>
constexpr int strided_threads(int logn, int loge) {
  if (loge < strided_loge<T, Op>()) return Op::kMulti ? 256 : 1024;
  return (sizeof(T) == 4 && Op::kMulti && logn <= 8 ? 4096 : strided_tile<T>()) >> loge;
}

// Register slot of a tile transform: slot number e (stable across calls),
// local line and position j + pr; pr is a constant of the slot (after
// unrolling), j the lane's own part: all of the position in mixed-radix
// tiles, below N / E (E elements per thread) and the same for every slot in
// power-of-two ones (tile_slot).
struct Slot {
  int e, line, j, pr;
  __host__ __device__ __forceinline__ int pos() const { return j + pr; }
};

// Radix of the stages of a length-2^LOGN transform with 2^LOGE elements per
// thread: as few stages as radices of at most 2^LOGE allow, the larger
// radices at the ends (1024 = 16 8 8 with 16 elements, 8 4 4 8 with 8).
template <int LOGN, int LOGE>
struct TilePlan {
  static constexpr int N = 1 << LOGN;
  static constexpr int E = 1 << LOGE;
  static constexpr int NS = (LOGN + LOGE - 1) / LOGE;
  static_assert(NS >= 1 && LOGE <= LOGN, "a thread's elements are of one line");
  static constexpr int lr(int s) {
    const int back = NS - 1 - s;
    const int rank = s <= back ? 2 * s : 2 * back + 1;
    return LOGN / NS + (rank < LOGN % NS ? 1 : 0);
  }
  static constexpr int lns(int s) {
    int n = 0;
    for (int i = 0; i < s; ++i) n += lr(i);
    return n;
  }
  // twiddle tables in LDS: entry [k R + r] = W_{Ns R}^{r k} of stage s >= 1
  static constexpr int twoff(int s) {
    int n = 0;
    for (int i = 1; i < s; ++i) n += 1 << lns(i + 1);
    return n;
  }
  static constexpr int NTW = twoff(NS);
};

// Slot e of stage S: butterfly j0 + (e / R) N / E, element e % R.
template <int LOGN, int LOGE, int S>
__host__ __device__ __forceinline__ Slot tile_slot(int e, int line, int j0) {
  using PL = TilePlan<LOGN, LOGE>;
  constexpr int R = 1 << PL::lr(S);
  return Slot{e, line, j0, (e % R) * (PL::N / R) + (e / R) * (PL::N / PL::E)};
}

// Copies the stages' twiddles to LDS from tw = exp(-2 pi i m / N).
template <typename T, int LOGN, int LOGE, int S = 1>
__device__ __forceinline__ void tile_twiddles(cpx<T>* s_tw, const cpx<T>* tw) {
  using PL = TilePlan<LOGN, LOGE>;
  if constexpr (S < PL::NS) {
    constexpr int lr = PL::lr(S), n = 1 << PL::lns(S + 1);
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
      const int k = i >> lr, r = i & ((1 << lr) - 1);
      s_tw[PL::twoff(S) + i] = tw[(r * k) << (LOGN - PL::lns(S + 1))];
    }
    tile_twiddles<T, LOGN, LOGE, S + 1>(s_tw, tw);
  }
}

// v[r] *= W^{r k} (conjugated for the inverse) from the stage's table row.
template <typename T, int DIR, int R>
__device__ __forceinline__ void tile_twiddle(cpx<T>* v, const cpx<T>* row) {
  cpx<T> w[R];
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int r = 0; r < R; r += 2) {
      const float4 q = *reinterpret_cast<const float4*>(row + r);
      w[r] = mk<T>(q.x, q.y);
      w[r + 1] = mk<T>(q.z, q.w);
    }
  } else {
#pragma unroll
    for (int r = 1; r < R; ++r) w[r] = row[r];
  }
#pragma unroll
  for (int r = 1; r < R; ++r) {
    const T wy = DIR > 0 ? -w[r].y : w[r].y;
    v[r] = mk<T>(fma_t(v[r].x, w[r].x, -(v[r].y * wy)), fma_t(v[r].x, wy, v[r].y * w[r].x));
  }
}

// Stages S .. of tile_fft_p2 (S >= 1): v holds stage S - 1's outputs.
template <typename T, int DIR, int LOGN, int LOGE, int S>
__device__ __forceinline__ void tile_stages(cpx<T> (&v)[1 << LOGE], cpx<T>* buf,
                                            const cpx<T>* s_tw, int logL, int j0, int line) {
  using PL = TilePlan<LOGN, LOGE>;
  constexpr int E = PL::E, N = PL::N;
  constexpr int lr = PL::lr(S), R = 1 << lr, NB = E / R;
  constexpr int lp = PL::lr(S - 1), Rp = 1 << lp, NBp = E / Rp;
  constexpr int Ns = 1 << PL::lns(S), Nsp = 1 << PL::lns(S - 1);
  // stage S - 1 writes position ((j - k) Rp + k) + r Nsp, stage S reads
  // j + r N / R: the fields of an address share no bit, so the pad of the
  // sum is the sum of the pads
  if constexpr (S > 1) __syncthreads();
#pragma unroll
  for (int i = 0; i < NBp; ++i) {
    const int j = j0 + i * (N / E);
    const int k = j & (Nsp - 1);
    const int a = lpad(((((j - k) << lp) + k) << logL) + line);
#pragma unroll
    for (int r = 0; r < Rp; ++r) buf[a + lpad((r * Nsp) << logL)] = v[i * Rp + r];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int a = lpad(((j0 + i * (N / E)) << logL) + line);
#pragma unroll
    for (int r = 0; r < R; ++r) v[i * R + r] = buf[a + lpad((r * (N / R)) << logL)];
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int k = (j0 + i * (N / E)) & (Ns - 1);
    tile_twiddle<T, DIR, R>(&v[i * R], s_tw + PL::twoff(S) + (k << lr));
    dftR<T, DIR, R>(&v[i * R]);
  }
  if constexpr (S + 1 < PL::NS)
    tile_stages<T, DIR, LOGN, LOGE, S + 1>(v, buf, s_tw, logL, j0, line);
}

// Full transform of one tile of 2^logL lines of length 2^LOGN by exactly
// N L / E threads (thread t: line t mod L, butterflies j = t / L + i N / E).
// src(slot) gives the inputs, dst(slot, v) receives the outputs,
// fetch(slot) is called for every first-stage slot once its input has been
// read: a multi-transform pass issues there the global loads of its next
// transform (same slots), in flight during this one's exchanges.  Ends with
// a barrier so buf can be reused (a length of at most E is one stage in
// registers and needs neither).
template <typename T, int DIR, int LOGN, int LOGE, class Src, class Dst, class Fetch>
__device__ __forceinline__ void tile_fft_p2(cpx<T>* buf, const cpx<T>* s_tw, int logL,
                                            Src&& src, Dst&& dst, const Fetch& fetch) {
  using PL = TilePlan<LOGN, LOGE>;
  constexpr int E = PL::E;
  const int line = threadIdx.x & ((1 << logL) - 1);
  const int j0 = threadIdx.x >> logL;
  constexpr int R0 = 1 << PL::lr(0);
  cpx<T> v[E];
#pragma unroll
  for (int e = 0; e < E; ++e)
    v[e] = src(tile_slot<LOGN, LOGE, 0>(e, line, j0));
#pragma unroll
  for (int i = 0; i < E / R0; ++i) dftR<T, DIR, R0>(&v[i * R0]);
#pragma unroll
  for (int e = 0; e < E; ++e)
    fetch(tile_slot<LOGN, LOGE, 0>(e, line, j0));
  if constexpr (PL::NS > 1) tile_stages<T, DIR, LOGN, LOGE, 1>(v, buf, s_tw, logL, j0, line);
#pragma unroll
  for (int e = 0; e < E; ++e) dst(tile_slot<LOGN, LOGE, PL::NS - 1>(e, line, j0), v[e]);
  if constexpr (PL::NS > 1) __syncthreads();
}

// Hook of tile_fft after the first stage (default: nothing).
struct NoFetch {
  __device__ __forceinline__ void operator()(const Slot&) const {}
};

template <typename T>
struct StridedDesc {
  int N;           // FFT length
  int L, logL;     // lines per tile (power of two)
  int nouter;      // number of independent planes
  int nlines;      // lines per plane
  int nf;          // fields transformed one after the other
  int kio;         // tiles remapped per XCD (K rows, or runs under a cache line)
  int stack;       // outputs of a line stacked as extra lines (OpYInv2NS)
  const cpx<T>* tw;  // exp(-2 pi i m / N), m < N
  // mixed-radix stages of a length without a power-of-two plan (gen_fft)
  int nst, inplace;
  int rad[kMaxStages];
};

// Full transform of one tile of 2^logL lines of length d.N.  LOGN > 0:
// power-of-two length (tile_fft_p2).  LOGN = 0: any length (gen_fft); slot
// e of both src and dst is the tile element threadIdx.x + e blockDim.x
// (line-fast), and the tile uses one or two LDS buffers (gen_fft).
template <typename T, int DIR, int LOGN, int LOGE, class Src, class Dst,
          class Fetch = NoFetch>
__device__ __forceinline__ void tile_fft(cpx<T>* buf, const cpx<T>* tw,
                                         const StridedDesc<T>& d, int logL, Src&& src,
                                         Dst&& dst, const Fetch& fetch = Fetch()) {
  if constexpr (LOGN > 0) {
    tile_fft_p2<T, DIR, LOGN, LOGE>(buf, tw, logL, src, dst, fetch);
  } else {
    constexpr int E = 1 << LOGE;
    const int tot = d.N << logL;
    const int lmask = (1 << logL) - 1;
    const TileLayout lay{1, (1 << logL) | 1};
    cpx<T>* A = buf;
    cpx<T>* B = d.inplace ? buf : buf + d.N * lay.sp;
    // all loads of a thread before the first use (slots past the tile repeat
    // its first element).  A tile of up to 256, 512 or 1024 elements runs one,
    // two or four slots only, as the source may be more than a load: a
    // Runge-Kutta step of ns2d on 48^2 83 -> 77 us in FP64 and 89 -> 77 in FP32,
    // on 100 x 200 103 -> 97 and 108 -> 96, of ns3d on 48^3 624 -> 565 and 545 ->
    // 359 us, against all 8 or 16 slots.
    auto in = [&](auto slots) {
      constexpr int n = decltype(slots)::value < E ? decltype(slots)::value : E;
      cpx<T> v[n];
#pragma unroll
      for (int e = 0; e < n; ++e) {
        const int idx = threadIdx.x + e * kGenThr, q = idx < tot ? idx : 0;
        v[e] = src(Slot{e, q & lmask, q >> logL, 0});
      }
#pragma unroll
      for (int e = 0; e < n; ++e) {
        const int idx = threadIdx.x + e * kGenThr;
        if (idx < tot) A[lay.at(idx & lmask, idx >> logL)] = v[e];
      }
#pragma unroll
      for (int e = 0; e < n; ++e) {
        const int idx = threadIdx.x + e * kGenThr, q = idx < tot ? idx : 0;
        fetch(Slot{e, q & lmask, q >> logL, 0});
      }
    };
    if (tot <= 1 * kGenThr)
      in(std::integral_constant<int, 1>());
    else if (tot <= 2 * kGenThr)
      in(std::integral_constant<int, 2>());
    else if (tot <= 4 * kGenThr)
      in(std::integral_constant<int, 4>());
    else
      in(std::integral_constant<int, E>());
    __syncthreads();
    const cpx<T>* res =
        gen_fft<T, DIR, kGenThr>(A, B, lay, tw, 1, d.N, 1 << logL, logL, d.nst, d.rad);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int idx = threadIdx.x + e * kGenThr;
      if (idx < tot)
        dst(Slot{e, idx & lmask, idx >> logL, 0}, res[lay.at(idx & lmask, idx >> logL)]);
    }
    __syncthreads();
  }
}

// Slot e of tile_fft's outputs; false where it holds none.
template <int LOGN, int LOGE, typename T>
__device__ __forceinline__ bool last_slot(int e, const StridedDesc<T>& d, int logL, Slot& s) {
  if constexpr (LOGN > 0) {
    s = tile_slot<LOGN, LOGE, TilePlan<LOGN, LOGE>::NS - 1>(
        e, (int)threadIdx.x & ((1 << logL) - 1), (int)threadIdx.x >> logL);
    return true;
  } else {
    const int idx = threadIdx.x + e * kGenThr;
    s = Slot{e, idx & ((1 << logL) - 1), idx >> logL, 0};
    return idx < (d.N << logL);
  }
}

// Lines of one side (input or output) of a tile: element (line, position p)
// of a field is at base[p' ps + line], p' = p - (p >= n - hi ? cut : 0).
// Positions in [lo, hi0) are zero when read and are not stored; lines from
// nl on neither.  cut > 0: the pruned positions are not in memory.
struct Lines {
  unsigned ps;
  int lo, hi0, cut, nl;
};

// all: nothing pruned.  A pruned axis of even length keeps at most n / 2
// non-negative positions (fsx_plan_create), so every position of the upper
// half belongs to the upper range.
__host__ __device__ __forceinline__ Lines lines_all(unsigned ps, int n, int nl) {
  return Lines{ps, n, 0, 0, nl};
}
__host__ __device__ __forceinline__ Lines lines_of(unsigned ps, const AxisMap& m, bool compact, int nl) {
  if (m.lo + m.hi == m.n) return lines_all(ps, m.n, nl);
  return Lines{ps, m.lo, m.n - m.hi, compact ? m.n - m.lo - m.hi : 0, nl};
}

// An integer the optimizer knows nothing about: comparisons with it stay
// selects (they would otherwise be threaded into branches around the loads,
// where a later test repeats them).
__host__ __device__ __forceinline__ int opaque(int x) {
#ifdef __HIP_DEVICE_COMPILE__
  asm("" : "+v"(x));
#endif
  return x;
}

// Holds n values in registers as they are: the last additions of a transform
// are otherwise sunk to the (conditional) uses of their results, and the
// butterfly's larger set of intermediate values stays live until then.
template <typename T, int E>
__device__ __forceinline__ void pin(cpx<T> (&v)[E]) {
#pragma unroll
  for (int e = 0; e < E; ++e) asm volatile("" : "+v"(v[e].x), "+v"(v[e].y));
}

// Whether slot s is kept on this side.  For power-of-two lengths lines past
// nl fail both comparisons through an out-of-range j.
template <int LOGN>
__host__ __device__ __forceinline__ bool ln_kept(const Lines& g, const Slot& s) {
  if constexpr (LOGN > 0) {
    constexpr int N = 1 << LOGN, H = N / 2;
    return s.pr >= H ? opaque(s.line < g.nl ? s.j : -N) >= g.hi0 - s.pr
                     : opaque(s.line < g.nl ? s.j : N) < g.lo - s.pr;
  } else {
    const int p = s.pos();
    return s.line < g.nl && (p < g.lo || p >= g.hi0);
  }
}
// Position offset of the slot's constant part (uniform; 64 bits).
template <int LOGN>
__host__ __device__ __forceinline__ long long ln_base(const Lines& g, const Slot& s) {
  constexpr int H = LOGN > 0 ? 1 << (LOGN - 1) : 1;
  return (long long)(s.pr >= H ? s.pr - g.cut : s.pr) * g.ps;
}
// Byte offset of the lane's part, in 32 bits: j and line only, so that it
// stays below lane_reach.
__host__ __device__ __forceinline__ unsigned ln_lane(const Lines& g, const Slot& s,
                                                     unsigned bytes) {
  return ((unsigned)s.j * g.ps + (unsigned)s.line) * bytes;
}
// Largest ln_lane of a power-of-two pass: n / E - 1 positions of pitch ps and
// the last of nl lines, values of `bytes` bytes.
inline unsigned long long lane_reach(int n, int loge, unsigned long long ps, int nl,
                                     unsigned bytes) {
  return (((unsigned long long)(n >> loge) - 1) * ps + (unsigned)(nl - 1)) * bytes;
}
// Small problems: power-of-two strided passes of fewer than kSmallWaves waves
// (4 per CU) with their usual 8 or 16 elements per thread give a thread 4
// (lengths 2^kSmallLogLo .. 2^kSmallLogHi).  A thread works through its
// modes one after the other (in the forward passes with a Runge-Kutta
// stage each has FP64 exponentials), and a pass of one wave per SIMD is as
// long as that chain.  A Runge-Kutta step of ns2d in a graph with 4 instead of
// 8 (FP64) or 16 (FP32) elements: 64^2 62 -> 54 us and 83 -> 54, 256^2 79 ->
// 71 and 96 -> 67, 512^2 100 -> 91 and 112 -> 81, 1024^2 FP32 (342 waves) 175
// -> 140; ns3d 64^3 175 -> 155 and 145 -> 128, 256 x 256 x 16 262 -> 228 and
// 203 -> 174 us.  With a limit of 256 waves the last two stay as they were.
// Fewer lines in a workgroup than fill a wave do not pay on top of that (64^3
// 155 -> 169 with 8 threads, 160 with 32): their rows are short runs.
constexpr int kSmallWaves = 1024;
constexpr int kSmallLogE = 2, kSmallLogLo = 4, kSmallLogHi = 10;
// log2 of the elements per thread of a length-2^logn pass over `lines` lines,
// given the usual one: fewer for a small problem, unless its lanes would reach
// too far for that (a mask that keeps next to nothing of a large field).
inline int small_loge(int logn, int loge, long long lines, unsigned long long ps,
                      unsigned bytes) {
  if (logn < kSmallLogLo || logn > kSmallLogHi || loge <= kSmallLogE) return loge;
  if (((lines << logn) >> loge) >= 64LL * kSmallWaves) return loge;
  // (a tile has at most 1024 lines)
  return lane_reach(1 << logn, kSmallLogE, ps, 1024, bytes) < kBufMax ? kSmallLogE : loge;
}
// Element offset of a slot (any length).
template <int LOGN>
__device__ __forceinline__ long long ln_offset(const Lines& g, const Slot& s) {
  if constexpr (LOGN > 0) {
    return ln_base<LOGN>(g, s) + (long long)s.j * g.ps + s.line;
  } else {
    const int p = s.pos();
    return (long long)(p >= g.lo ? p - g.cut : p) * g.ps + s.line;
  }
}
template <int LOGN, typename T>
__device__ __forceinline__ cpx<T> ln_load(const Lines& g, const cpx<T>* base, const Slot& s) {
  if constexpr (LOGN > 0) {
    const unsigned off = ln_lane(g, s, sizeof(cpx<T>));
    return buf_load<T>(buf_rsrc(base + ln_base<LOGN>(g, s), kBufMax),
                       ln_kept<LOGN>(g, s) ? off : kOOB);
  } else {
    // element 0 is read in place of a masked one: no branch around the load
    const bool ok = ln_kept<LOGN>(g, s);
    const cpx<T> v = base[ok ? ln_offset<LOGN>(g, s) : 0];
    return ok ? v : zero<T>();
  }
}
template <int LOGN, typename T>
__device__ __forceinline__ void ln_store(const Lines& g, cpx<T>* base, const Slot& s, cpx<T> v) {
  if constexpr (LOGN > 0) {
    const unsigned off = ln_lane(g, s, sizeof(cpx<T>));
    buf_store<T>(buf_rsrc(base + ln_base<LOGN>(g, s), kBufMax),
                 ln_kept<LOGN>(g, s) ? off : kOOB, v);
  } else {
    if (ln_kept<LOGN>(g, s)) base[ln_offset<LOGN>(g, s)] = v;
  }
}
// Whether a stored mode is dealiased by the mask (laid out like the field).
template <int LOGN>
__device__ __forceinline__ bool ln_masked(const Lines& g, const unsigned char* mask,
                                          const Slot& s) {
  return mask && ln_kept<LOGN>(g, s) && mask[ln_offset<LOGN>(g, s)] != 0;
}

// Mode of a slot in the state arrays, for rk_point.
template <int LOGN, typename T>
struct SlotMode {
  const Lines& g;
  const Slot& s;
  long long base;
  __device__ __forceinline__ cpx<T> load(const cpx<T>* a) const {
    return ln_load<LOGN, T>(g, a + base, s);
  }
  __device__ __forceinline__ void store(cpx<T>* a, cpx<T> v) const {
    ln_store<LOGN, T>(g, a + base, s, v);
  }
};

}  // namespace fsx

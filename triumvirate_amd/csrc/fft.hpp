// fft.hpp -- 3-D complex FFT for gfx950: three batched 1-D passes, each a
// radix-4 Stockham autosort transform (the formulation of Govindaraju et
// al., "High performance discrete Fourier transforms on graphics
// processors", SC 2008) held in registers, eight elements of a line per
// thread, with one exchange through LDS between its stages.
//
// Sizes: powers of two from 8 to 1024 per axis.  Sign convention as FFTW
// (forward e^{-ikx}, backward e^{+ikx}), unnormalised.
//
// Each pass is in place: a workgroup takes whole lines of one axis, every
// thread loads its eight elements, transforms them and writes them back to
// the same addresses, so no second buffer is needed.  The first pass takes a
// "loader" functor that produces each input element from one or more source
// fields; shell filters, window deconvolution, scalings and two-point
// products are fused there instead of costing a separate read+write sweep of
// the mesh.
#pragma once

#include "common.hpp"

namespace trvg {

constexpr int FFT_THREADS = 256;


// Global stores and loads of the passes' mesh data (one place for their
// cache policy; plain accesses measured best: streaming hints gained on
// some passes and lost on others).
template <typename T>
__device__ __forceinline__ void st_mesh(c2<T>* p, c2<T> v) { *p = v; }

template <typename T>
__device__ __forceinline__ c2<T> ld_mesh(const c2<T>* p) { return *p; }

// Workgroups are dispatched to the 8 XCDs round-robin by index; mapping
// index b to logical block (b % 8) * (n / 8) + b / 8 gives each XCD (and
// its L2) a contiguous range of blocks, so neighbouring blocks that share
// cache lines run under one L2.  Identity when n is not a multiple of 8.
__device__ __forceinline__ long long xcd_block(long long b, long long n) {
  if (n % 8 != 0) return b;
  return (b % 8) * (n / 8) + b / 8;
}

// Support pruning for band-limited inverse transforms: input cells exist only
// where |k| < k_hi, so (with kcut2 = k_hi^2 (1 + 1e-9))
//   line (i, j) of the z pass is needed only if kx^2 + ky^2 < kcut2 (P1);
//   slab i of the y pass only if kx^2 < kcut2 (P2).
// Passes skip what is not needed, and later passes read only rows that
// earlier passes wrote, treating the rest as zero.
struct Prune {
  int on;
  double kcut2;
  double dk0, dk1;
  int n0, n1;
  // Explicitly rounded operations: every pass must evaluate the predicates
  // identically (no contraction differences between kernels).
  __device__ __forceinline__ bool p2(int i) const {
    double kx = __dmul_rn(double(shifted(i, n0)), dk0);
    return __dmul_rn(kx, kx) < kcut2;
  }
  // Largest |m| of a row index m with P1(i, m) (reach_j; -1: none), or with
  // P2(m) (reach_i): the predicates fall with |m|, so rows compare as integers.
  // Estimated in FP32 and settled by the predicate itself.
  __device__ __forceinline__ int reach_j(int i) const {
    const double kx = __dmul_rn(double(shifted(i, n0)), dk0);
    return reach(__dmul_rn(kx, kx), dk1, n1 / 2);
  }
  __device__ __forceinline__ int reach_i() const { return reach(0., dk0, n0 / 2); }
  __device__ __forceinline__ int reach(double k2, double dk, int top) const {
    auto in = [&](int m) {
      const double k = __dmul_rn(double(m), dk);
      return __dadd_rn(k2, __dmul_rn(k, k)) < kcut2;
    };
    const float f = sqrtf(fmaxf(float(kcut2 - k2), 0.f)) / float(dk);
    int m = f < float(top) ? int(f) : top;
    while (m < top && in(m + 1)) m++;
    while (m >= 0 && !in(m)) m--;
    return m;
  }
  __device__ __forceinline__ bool p1(int i, int j) const {
    double kx = __dmul_rn(double(shifted(i, n0)), dk0);
    double ky = __dmul_rn(double(shifted(j, n1)), dk1);
    return __dadd_rn(__dmul_rn(kx, kx), __dmul_rn(ky, ky)) < kcut2;
  }
};

// ---------------------------------------------------------------------------
// Register-resident DFTs.
// ---------------------------------------------------------------------------

// cos and sin of 2 pi k / p at compile time (Taylor series about 0 after
// reduction to |x| <= pi).
constexpr double cx_series(double x, bool odd) {
  double term = odd ? x : 1., sum = term;
  for (int i = odd ? 2 : 1; i < 60; i += 2) {
    term *= -x * x / (double(i) * double(i + 1));
    sum += term;
  }
  return sum;
}
constexpr double cx_turn(int k, int p) {
  const int r = k % p;
  return 2. * 3.14159265358979323846 * double(2 * r > p ? r - p : r) / double(p);
}

// d * e^{sgn i pi k / 4} for k in [0, 4); k is a constant after unrolling, so
// the trivial factors (1, +-i) cost no multiplications.  FP32: cos pi / 4 in two
// parts, as the twiddles below.
template <typename T>
__device__ __forceinline__ c2<T> rot_pi4(c2<T> d, int k, T sgn) {
  if (k == 0) return d;
  const c2<T> r = mk<T>(-sgn * d.y, sgn * d.x);   // d * sgn i
  if (k == 2) return r;
  const c2<T> s = k == 1 ? cadd<T>(d, r) : csub<T>(r, d);
  constexpr T c = T(0.70710678118654752440);
  constexpr T l = T(0.70710678118654752440 - double(c));
  if (sizeof(T) == 4) return mk<T>(s.x * c + s.x * l, s.y * c + s.y * l);
  return mk<T>(s.x * c, s.y * c);
}

// One decimation-in-frequency radix-2 stage of length LEN over v[0, R),
// then the stages of length LEN / 2 ... 2.
template <typename T, int R, int LEN>
struct DifStages {
  static __device__ __forceinline__ void run(c2<T>* v, T sgn) {
    constexpr int H = LEN / 2;
#pragma unroll
    for (int s = 0; s < R; s += LEN) {
#pragma unroll
      for (int j = 0; j < H; j++) {
        const c2<T> a = v[s + j], b = v[s + j + H];
        v[s + j] = cadd<T>(a, b);
        v[s + j + H] = rot_pi4<T>(csub<T>(a, b), (8 / LEN) * j, sgn);
      }
    }
    DifStages<T, R, H>::run(v, sgn);
  }
};
template <typename T, int R>
struct DifStages<T, R, 1> {
  static __device__ __forceinline__ void run(c2<T>*, T) {}
};

__host__ __device__ constexpr int bitrev(int k, int bits) {
  return bits == 0 ? 0 : ((k & 1) << (bits - 1)) | bitrev(k >> 1, bits - 1);
}
__host__ __device__ constexpr int ilog2c(int r) { return r <= 1 ? 0 : 1 + ilog2c(r / 2); }

// v <- DFT_R(v): X[k] = sum_n v[n] e^{sgn 2 pi i n k / R}, natural order in
// and out (R a power of two <= 8, held in registers).
template <typename T, int R>
__device__ __forceinline__ void dft_reg(c2<T>* v, T sgn) {
  static_assert(R >= 1 && R <= 8 && (R & (R - 1)) == 0, "register DFT size");
  DifStages<T, R, R>::run(v, sgn);
  c2<T> o[R];
#pragma unroll
  for (int k = 0; k < R; k++) o[k] = v[bitrev(k, ilog2c(R))];
#pragma unroll
  for (int k = 0; k < R; k++) v[k] = o[k];
}

// ---------------------------------------------------------------------------
// Line transforms: N = 2^LOGN points as stages of radix 2^LR, the last one of
// what is left.  Thread j < N / 8 of a line holds its elements j + e N / 8,
// e < 8, before and after (so global accesses of neighbouring threads are
// adjacent at both ends); between two stages the line goes through LDS once.
//
// Bound by HBM (80-90 % of the copy rate) where the mesh exceeds the caches.
// Against radix-4 stages with the line in LDS throughout, a transform
// crosses LDS 6 times instead of 10 (N = 256), starts from the loads
// themselves and ends in the stores, and masked rows are loaded together
// instead of one after the other.  Radix 4 (51 registers in FP32, 72 in
// FP64 for N = 256: eight and seven waves per SIMD) beats radix 8 (90 and
// 126), whose fewer exchanges do not make up for the waves.  Measured,
// before and after, in us: strided pass of 256^3 FP32 63 -> 48, FP64 103 ->
// 86, of 512^3 FP32 698 -> 455; y pass of 30 FP32 fields of 512^3 17.0 ->
// 12.3 ms; masked z pass of the same 17.6 -> 11.6 ms (there against a
// register transform of 16 x 32 points), of 12.5 FP64 fields of 256^3 849 ->
// 574 us.  Twiddles in two parts (below) add 1 to 7 % to FP32 passes.
// ---------------------------------------------------------------------------

// Log2 of the radix of the stages.
constexpr int FFT_LR = 2;

// LDS position of element n: one element of padding per eight, which spreads
// the writes of the first stage (stride 4, or 8 of radix-8 stages) over all
// banks.
__host__ __device__ __forceinline__ constexpr int fft_pad(int n) { return n + n / 8; }

// LDS elements between the lines of a workgroup: nl lanes in a row belong to
// different lines (1: to the same), and are kept on different banks.
template <typename T>
constexpr int fft_line_stride(int n, int nl) {
  const int banks = 128 / int(sizeof(c2<T>));   // elements across the banks
  const int base = fft_pad(n);
  if (nl == 1) return base;
  const int want = nl >= banks ? 1 : banks / nl;
  return base + ((want - base) % banks + banks) % banks;
}

// FP32 twiddles of the stages up to span 16 are kept in two parts: these stages
// use a handful of angles (multiples of 2 pi / 64) over and over, so that their
// rounding scales every mode alike (e^{i pi / 4} alone is short by 1.7e-8)
// and does not average out over a mesh.  With single parts a transform of 64^3
// to 256^3 comes out short by 6e-8, a bispectrum by 1.8e-7; with both parts by
// less than 3e-9 and 2 to 4e-8.  Strided pass of 256^3 42.5 -> 43.8 us, z pass 48.8
// -> 52.0.  Second parts of cos and sin 2 pi m / 64:
constexpr int FFT_LO = 64;
struct TwiddleLo {
  float2 v[FFT_LO];
};
constexpr TwiddleLo make_twiddle_lo() {
  TwiddleLo t{};
  for (int m = 0; m < FFT_LO; m++) {
    const double c = cx_series(cx_turn(m, FFT_LO), false), s = cx_series(cx_turn(m, FFT_LO), true);
    t.v[m].x = float(c - double(float(c)));
    t.v[m].y = float(s - double(float(s)));
  }
  return t;
}
static __device__ const TwiddleLo twiddle_lo = make_twiddle_lo();

// x w, and for FP32 the second part l of w.
template <typename T>
__device__ __forceinline__ c2<T> tw_mul(c2<T> x, c2<T> w, c2<T> l) {
  return mk<T>(fma(x.x, w.x, fma(-x.y, w.y, fma(x.x, l.x, -x.y * l.y))),
               fma(x.x, w.y, fma(x.y, w.x, fma(x.x, l.y, x.y * l.x))));
}

// Twiddles in LDS, per stage (span Ns, radix R) the (R - 1) Ns factors
// w^{q k N / (Ns R)}, k fastest: N - 2^LR of them (the spans add up so).  tw:
// e^{sign 2 pi i m / N}.
template <typename T>
__device__ __forceinline__ void fft_fill_lo(c2<T>* lo, int t, T sgn) {
  if constexpr (sizeof(T) == 4) {
    if (t < FFT_LO) lo[t] = mk<T>(twiddle_lo.v[t].x, sgn * twiddle_lo.v[t].y);
  }
}
template <typename T, int LOGN, int LR = FFT_LR, int LD = LR>
__device__ __forceinline__ void fft_fill_twiddles(c2<T>* W, const c2<T>* __restrict__ tw,
                                                  int t, int nt) {
  if constexpr (LD < LOGN) {
    constexpr int N = 1 << LOGN, Ns = 1 << LD;
    constexpr int R = 1 << (LOGN - LD >= LR ? LR : LOGN - LD);
    for (int i = t; i < (R - 1) * Ns; i += nt) {
      const int q = i / Ns + 1, k = i % Ns;
      W[i] = tw[q * k * (N / (Ns * R))];
    }
    fft_fill_twiddles<T, LOGN, LR, LD + LR>(W + (R - 1) * Ns, tw, t, nt);
  }
}

// Stages from span 2^LD on.  `lb`: this line in LDS.  WAVE: the line's
// threads are one wave's, which needs no barrier.  AGAIN: LDS may still be
// read by an earlier transform of the workgroup.
template <typename T, int LOGN, int LR, bool WAVE, bool AGAIN, int LD = 0>
__device__ __forceinline__ void fft_stages(c2<T> (&v)[8], c2<T>* lb, const c2<T>* W,
                                           const c2<T>* lo, int j, T sgn) {
  constexpr int N = 1 << LOGN, M = N / 8, Ns = 1 << LD;
  constexpr int R = 1 << (LOGN - LD >= LR ? LR : LOGN - LD);
  constexpr int NB = 8 / R;                 // butterflies per thread
  constexpr bool LAST = LD + LR >= LOGN;
  auto sync = [] {
    if (WAVE) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
      __syncthreads();
    }
  };
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const int jb = j + b * M, k = jb & (Ns - 1);
    c2<T> x[R];
#pragma unroll
    for (int q = 0; q < R; q++) {
      x[q] = v[b + q * NB];
      if (LD > 0 && q > 0) {
        const c2<T> w = W[(q - 1) * Ns + k];
        if constexpr (sizeof(T) == 4 && Ns <= 16) x[q] = tw_mul<T>(x[q], w, lo[q * k * (FFT_LO / (Ns * R))]);
        else x[q] = cmul<T>(x[q], w);
      }
    }
    dft_reg<T, R>(x, sgn);
#pragma unroll
    for (int r = 0; r < R; r++) v[b + r * NB] = x[r];
  }
  if constexpr (!LAST) {
    if (LD > 0 || AGAIN) sync();
#pragma unroll
    for (int b = 0; b < NB; b++) {
      const int jb = j + b * M, k = jb & (Ns - 1);
      const int d = (jb / Ns) * (Ns * R) + k;
#pragma unroll
      for (int r = 0; r < R; r++) lb[fft_pad(d + r * Ns)] = v[b + r * NB];
    }
    sync();
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = lb[fft_pad(j + e * M)];
    fft_stages<T, LOGN, LR, WAVE, AGAIN, LD + LR>(v, lb, LD > 0 ? W + (R - 1) * Ns : W, lo, j, sgn);
  }
}

// LDS of a workgroup: nl lines (stride `ls`) and the twiddles of its stages,
// n minus the first radix of them at most.
constexpr size_t FFT_LDS = 160 * 1024;
template <typename T>
constexpr size_t fft_lds(int n, int nl, int ls) {
  return size_t(nl * ls + n - (1 << FFT_LR)) * sizeof(c2<T>) +
         (sizeof(T) == 4 ? FFT_LO * sizeof(float2) : 0);
}
template <typename T>
constexpr size_t strided_lds(int logn, int nt) {
  const int nl = nt * 8 >> logn;
  return fft_lds<T>(1 << logn, nl, fft_line_stride<T>(1 << logn, nl));
}

// Threads of a workgroup of the strided passes: rows of `bytes` contiguous
// bytes (several lines of neighbouring columns), within 256..1024 threads.
// From 512 points on 256 threads would hold rows of 32 bytes, half a sector
// of HBM; up to 256 points rows of 64 bytes measured no slower than 128, and
// the smaller blocks prune better.  Eight FP64 lines of 1024 points do not
// fit LDS: rows of 64 bytes there (x pass of 1024 x 512 x 256: 2.06 ms; rows
// of 32 bytes 2.20).
template <typename T, int LOGN>
constexpr int strided_threads() {
  const int bytes = LOGN >= 9 ? 128 : 64;
  int nt = bytes / int(sizeof(c2<T>)) * ((1 << LOGN) / 8);
  nt = nt < 256 ? 256 : (nt > 1024 ? 1024 : nt);
  while (strided_lds<T>(LOGN, nt) > FFT_LDS) nt /= 2;
  return nt;
}
template <typename T, int LOGN>
constexpr int strided_lines() { return strided_threads<T, LOGN>() * 8 >> LOGN; }
template <typename T, int LOGN>
constexpr size_t strided_smem() {
  constexpr size_t bytes = strided_lds<T>(LOGN, strided_threads<T, LOGN>());
  static_assert(bytes <= FFT_LDS, "lines of a strided workgroup exceed LDS");
  return bytes;
}
// Lines of a workgroup of the z pass (256 threads).
constexpr int z_lines(int n) { return FFT_THREADS * 8 / n; }
template <typename T, int LOGN>
constexpr size_t z_smem() {
  constexpr int N = 1 << LOGN;
  constexpr size_t bytes = fft_lds<T>(N, z_lines(N), fft_line_stride<T>(N, 1));
  static_assert(bytes <= FFT_LDS, "lines of a z workgroup exceed LDS");
  return bytes;
}

// Loaders that read several fields or evaluate harmonics per cell.
template <class Loader> struct HeavyLoader { static constexpr bool value = false; };

// First pass along z (contiguous lines), with a fused loader, for block
// `blk` of the mesh at `data` (z_lines(N) lines; the last block of a mesh may
// hold fewer of its nlines).
// Loader: c2<T> operator()(long long g, int i, int j, int k) const.
template <typename T, int LOGN, class Loader>
__device__ __forceinline__ void fft_z_block(c2<T>* __restrict__ data, const Loader& load,
                                            const c2<T>* __restrict__ tw, int n1,
                                            long long nlines, int sign, const Prune& pr,
                                            long long blk) {
  constexpr int N = 1 << LOGN, M = N / 8;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  constexpr int LS = fft_line_stride<T>(N, 1);
  c2<T>* buf = reinterpret_cast<c2<T>*>(smem_raw);
  c2<T>* W = buf + z_lines(N) * LS;
  const int t = threadIdx.x, l = t / M, j = t % M;
  // Threads past the last line repeat it and do not write (loads without a
  // branch stay in flight together).
  const bool valid = blk * z_lines(N) + l < nlines;
  const long long line = valid ? blk * z_lines(N) + l : nlines - 1;
  const int i1 = int(unsigned(line) / unsigned(n1)), j1 = int(unsigned(line) % unsigned(n1));
  if (pr.on) {
    // Skip the workgroup if none of its lines is needed (uniform exit).
    bool any = false;
    for (int q = 0; q < z_lines(N) && !any; q++) {
      const long long ln = blk * z_lines(N) + q;
      any = ln < nlines && pr.p1(int(ln / n1), int(ln % n1));
    }
    if (!any) return;
  }
  c2<T>* lo = W + N - (1 << FFT_LR);
  fft_fill_twiddles<T, LOGN>(W, tw, t, FFT_THREADS);
  fft_fill_lo<T>(lo, t, T(sign));
  c2<T> v[8];
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const int k = j + e * M;
    v[e] = load(line * N + k, i1, j1, k);
    // Loaders with per-cell arithmetic: four cells at a time, which keeps the
    // registers (and with them the waves) of the pass within bounds.
    if (HeavyLoader<Loader>::value && e % 4 == 3) __builtin_amdgcn_sched_barrier(0);
  }
  if (M <= 64) __syncthreads();   // the twiddles; the stages stay within a wave
  fft_stages<T, LOGN, FFT_LR, (M <= 64), false>(v, buf + l * LS, W, lo, j, T(sign));
  if (!valid) return;
  c2<T>* out = data + line * N + j;
#pragma unroll
  for (int e = 0; e < 8; e++) st_mesh<T>(out + e * M, v[e]);
}

template <typename T, int LOGN, class Loader>
__global__ void __launch_bounds__(FFT_THREADS)
fft_pass_z(c2<T>* __restrict__ data, Loader load, const c2<T>* __restrict__ tw,
           int n1, long long nlines, int sign, Prune pr) {
  fft_z_block<T, LOGN>(data, load, tw, n1, nlines, sign, pr, xcd_block(blockIdx.x, gridDim.x));
}

// Batched first pass over several fields (a slab of meshes `fstride` apart):
// work[b] = (field, block) lists only the blocks with needed lines, so
// blocks outside every band cost nothing.  BatchLoader::field(q) returns
// the loader of field q; kcut2[q] is that field's pruning radius.
template <typename T, int LOGN, class BatchLoader>
__global__ void __launch_bounds__(FFT_THREADS)
fft_pass_z_batch(c2<T>* __restrict__ base, long long fstride, BatchLoader load,
                 const c2<T>* __restrict__ tw, int n1, long long nlines, int sign, Prune pr,
                 const double* __restrict__ kcut2, const int2* __restrict__ work) {
  const int2 wk = work[xcd_block(blockIdx.x, gridDim.x)];
  Prune p = pr;
  p.kcut2 = kcut2[wk.x];
  fft_z_block<T, LOGN>(base + wk.x * fstride, load.field(wk.x), tw, n1, nlines, sign, p, wk.y);
}

// Strided pass: lines of length N with element stride S.  Line `id` starts
// at (id / inner) * outer_stride + id % inner, so consecutive lines are
// adjacent in memory within a slice:
//   y pass: S = n2, inner = n2, outer_stride = n1*n2;
//   x pass: S = n1*n2, inner = n1*n2, outer_stride = 0.
// Each workgroup takes strided_lines consecutive lines (the last fewer).
//
// prune_mode (with pr.on): 1 = y pass (slab i = id / inner must satisfy P2,
// row j read only where P1(i, j)); 2 = x pass (row i read only where P2(i));
// 3 = y pass of the x-first order (Prune over the (z, y) axes: line k =
// id % inner written only where P2(k), row j read only where P1(k, j)).
template <typename T, int LOGN>
__device__ __forceinline__ void fft_strided_block(
    c2<T>* __restrict__ data, const c2<T>* __restrict__ tw, long long S,
    long long outer_stride, long long inner, long long nlines, int sign, const Prune& pr,
    int prune_mode, long long blk) {
  constexpr int N = 1 << LOGN, M = N / 8;
  constexpr int NL = strided_lines<T, LOGN>();
  constexpr int LS = fft_line_stride<T>(N, NL);
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  c2<T>* buf = reinterpret_cast<c2<T>*>(smem_raw);
  c2<T>* W = buf + NL * LS;
  const int t = threadIdx.x, l = t % NL, j = t / NL;
  const bool valid = blk * NL + l < nlines;
  const long long id = valid ? blk * NL + l : nlines - 1;
  // Line counts fit 32 bits (axes up to 2048).
  const unsigned in = unsigned(inner), slice = unsigned(id) / in, col = unsigned(id) % in;
  bool line_in = valid;
  if (pr.on && prune_mode != 2) {
    bool any = false;   // uniform exit when no line is needed
    for (int q = 0; q < NL && !any; q++) {
      const unsigned ln = unsigned(blk * NL + q);
      any = ln < nlines && pr.p2(int(prune_mode == 1 ? ln / in : ln % in));
    }
    if (!any) return;
    line_in = valid && pr.p2(int(prune_mode == 1 ? slice : col));
  }
  c2<T>* lo = W + N - (1 << FFT_LR);
  fft_fill_twiddles<T, LOGN>(W, tw, t, strided_threads<T, LOGN>());
  fft_fill_lo<T>(lo, t, T(sign));
  c2<T>* p = data + (long long)slice * outer_stride + col + (long long)j * S;
  const long long step = (long long)M * S;
  c2<T> v[8];
  if (pr.on) {
    const int reach =
        !line_in ? -1 : (prune_mode == 2 ? pr.reach_i() : pr.reach_j(int(prune_mode == 1 ? slice : col)));
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const int m = shifted(j + e * M, N);
      v[e] = (m < 0 ? -m : m) <= reach ? ld_mesh<T>(p + e * step) : mk<T>(T(0), T(0));
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = ld_mesh<T>(p + e * step);
  }
  fft_stages<T, LOGN, FFT_LR, false, false>(v, buf + l * LS, W, lo, j, T(sign));
  if (!line_in) return;
#pragma unroll
  for (int e = 0; e < 8; e++) st_mesh<T>(p + e * step, v[e]);
}

template <typename T, int LOGN>
__global__ void __launch_bounds__((strided_threads<T, LOGN>()))
fft_pass_strided(c2<T>* __restrict__ data, const c2<T>* __restrict__ tw,
                 long long S, long long outer_stride, long long inner, long long nlines,
                 int sign, Prune pr, int prune_mode) {
  fft_strided_block<T, LOGN>(data, tw, S, outer_stride, inner, nlines, sign, pr, prune_mode,
                             xcd_block(blockIdx.x, gridDim.x));
}

// Batched strided pass over a slab of fields, work[b] = (field, block).
template <typename T, int LOGN>
__global__ void __launch_bounds__((strided_threads<T, LOGN>()))
fft_pass_strided_batch(c2<T>* __restrict__ base, long long fstride,
                       const c2<T>* __restrict__ tw, long long S,
                       long long outer_stride, long long inner, long long nlines, int sign,
                       Prune pr, const double* __restrict__ kcut2,
                       const int2* __restrict__ work, int prune_mode) {
  const int2 wk = work[xcd_block(blockIdx.x, gridDim.x)];
  Prune p = pr;
  p.kcut2 = kcut2[wk.x];
  fft_strided_block<T, LOGN>(base + wk.x * fstride, tw, S, outer_stride, inner, nlines, sign,
                             p, prune_mode, wk.y);
}

// First pass of the x-first order: lines along x (length N = n0, element
// stride S = n1 n2), line id = j n2 + k, with a fused loader
// load(g, i, j, k).  Prune over the (z, y) axes: a block runs only if one of
// its lines has P1(k, j), and only those lines are written (the y pass
// reads no other).
template <typename T, int LOGN, class Loader>
__device__ __forceinline__ void fft_x_load_block(c2<T>* __restrict__ data,
                                                 const Loader& load,
                                                 const c2<T>* __restrict__ tw,
                                                 int n1, int n2, int sign,
                                                 const Prune& pr, long long blk) {
  constexpr int N = 1 << LOGN, M = N / 8;
  constexpr int NL = strided_lines<T, LOGN>();
  constexpr int LS = fft_line_stride<T>(N, NL);
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  c2<T>* buf = reinterpret_cast<c2<T>*>(smem_raw);
  c2<T>* W = buf + NL * LS;
  const int t = threadIdx.x, l = t % NL, r0 = t / NL;
  const long long S = (long long)n1 * n2;
  const long long id = blk * NL + l;
  const int j = int(unsigned(id) / unsigned(n2)), k = int(unsigned(id) % unsigned(n2));
  bool line_in = id < S;
  if (pr.on) {
    bool any = false;   // uniform exit when no line is needed
    for (int q = 0; q < NL && !any; q++) {
      const unsigned ln = unsigned(blk * NL + q);
      any = ln < S && pr.p1(int(ln % unsigned(n2)), int(ln / unsigned(n2)));
    }
    if (!any) return;
    line_in = line_in && pr.p1(k, j);
  }
  c2<T>* lo = W + N - (1 << FFT_LR);
  fft_fill_twiddles<T, LOGN>(W, tw, t, strided_threads<T, LOGN>());
  fft_fill_lo<T>(lo, t, T(sign));
  c2<T> v[8];
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const int n = r0 + e * M;
    v[e] = line_in ? load(id + (long long)n * S, n, j, k) : mk<T>(T(0), T(0));
    if (HeavyLoader<Loader>::value && e % 4 == 3) __builtin_amdgcn_sched_barrier(0);
  }
  fft_stages<T, LOGN, FFT_LR, false, false>(v, buf + l * LS, W, lo, r0, T(sign));
  if (!line_in) return;
#pragma unroll
  for (int e = 0; e < 8; e++) st_mesh<T>(data + id + (long long)(r0 + e * M) * S, v[e]);
}

// Batched x-first loader pass, work[b] = (field, block).
template <typename T, int LOGN, class BatchLoader>
__global__ void __launch_bounds__((strided_threads<T, LOGN>()))
fft_pass_x_load_batch(c2<T>* __restrict__ base, long long fstride, BatchLoader load,
                      const c2<T>* __restrict__ tw, int n1, int n2, int sign, Prune pr,
                      const double* __restrict__ kcut2, const int2* __restrict__ work) {
  const int2 wk = work[xcd_block(blockIdx.x, gridDim.x)];
  Prune p = pr;
  p.kcut2 = kcut2[wk.x];
  fft_x_load_block<T, LOGN>(base + wk.x * fstride, load.field(wk.x), tw, n1, n2, sign, p,
                            wk.y);
}

// Identity loader (plain in-place transform).
template <typename T>
struct LoadSame {
  const c2<T>* src;
  __device__ c2<T> operator()(long long g, int, int, int) const {
    return ld_mesh<T>(src + g);
  }
};

}  // namespace trvg

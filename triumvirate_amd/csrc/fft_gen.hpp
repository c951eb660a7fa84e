// fft_gen.hpp -- FFT passes for mesh axes that are not powers of two.
//
// An axis of length N (even, N <= 2048) is transformed in LDS by a
// mixed-radix Stockham sequence N = r_0 r_1 ... (radix 4 while it divides,
// then 2, then the odd primes in ascending order).  Stage s with span
// Ns = r_0 ... r_{s-1} and radix p takes butterfly j < N / p, k = j mod Ns,
//   out[(j / Ns) Ns p + k + r Ns] = sum_q in[j + q N/p] w^{q (k N/(Ns p) + r N/p)},
// r < p, w = e^{sign 2 pi i / N}.  Radices up to 7 are butterflies in
// registers over one LDS buffer (read, barrier, write back); a length with a
// larger prime factor forms every output directly, reading one buffer and
// writing another (any prime radix works; a radix-p stage costs p products
// per output).  Sign convention and normalisation as the power-of-two passes
// (FFTW's, unnormalised).
//
// A workgroup takes NL = max(1, 2048 / N) lines of one axis (the last block
// of an axis may hold fewer); the passes mirror those of fft.hpp: the z pass
// with a loader, the strided passes with the same pruning modes, the x-first
// loader pass and the j_l multi-field x pass, each also over (field, block)
// work lists.
//
// FP32 lines are FP32 in memory and LDS, but their register butterflies are
// formed in FP64, with FP64 twiddles.  A rounded constant (a twiddle, cos 2 pi
// / 5) is the same for every line, so its error does not average out over a
// mesh as that of rounded data does: with FP32 butterflies an FP32 window
// function of 96^3 was off by 1.7e-7 (every output formed directly: 1.2e-7),
// with FP64 ones by 2.2e-8.  FP64 products issue at the rate of FP32 ones; the
// strided pass of 200^3 FP32 takes 62 us (FP32 butterflies 51, every output
// formed directly 142).
//
// What bounded them: integer divisions (three or more per element, some in
// 64 bits, and four per output of every stage) and p LDS reads per output.
// Indexes now come from one multiplication with a reciprocal of the plan,
// elements are loaded eight at a time, and one buffer instead of two holds
// twice the workgroups per CU.  200^3 FP64: strided pass 218 -> 69 us (3.7 TB/s),
// z pass 196 -> 59 us.
#pragma once

#include "fft.hpp"

namespace trvg {

constexpr int GEN_ELEMS = FFT_THREADS * 8;   // target elements per workgroup
constexpr int GEN_MAX_N = 2048;
constexpr int GEN_MAX_STAGES = 16;

constexpr int GEN_MAXE = GEN_ELEMS / FFT_THREADS;   // elements per thread

// floor(x / d) for x, d below 2^16 by one multiplication.
struct GenDiv {
  unsigned d, m;   // m = ceil(2^32 / d); d = 1: m = 0
  __device__ __forceinline__ int div(int x) const {
    return d == 1 ? x : int(__umulhi(unsigned(x), m));
  }
};

struct GenPlan {
  int n;      // line length
  int nl;     // lines per workgroup
  int nst;    // stages
  int direct; // a prime factor above 7: outputs formed directly, two buffers
  int radix[GEN_MAX_STAGES];
  GenDiv by_n, by_nl;                 // by n, by nl
  GenDiv by_np[GEN_MAX_STAGES];       // by n / radix
  GenDiv by_ns[GEN_MAX_STAGES];       // by the span
};

inline int gen_lines_per_block(int n) { return n <= GEN_ELEMS ? GEN_ELEMS / n : 1; }

inline GenDiv make_gen_div(int d) {
  const unsigned long long m = ((1ull << 32) + unsigned(d) - 1) / unsigned(d);
  return GenDiv{unsigned(d), d == 1 ? 0u : unsigned(m)};
}

inline GenPlan make_gen_plan(int n) {
  GenPlan p{};
  p.n = n;
  p.nl = gen_lines_per_block(n);
  int m = n, ns = 1;
  auto push = [&](int r) {
    p.by_np[p.nst] = make_gen_div(n / r);
    p.by_ns[p.nst] = make_gen_div(ns);
    p.radix[p.nst++] = r;
    p.direct |= r > 7;
    ns *= r;
  };
  while (m % 4 == 0) { push(4); m /= 4; }
  while (m % 2 == 0) { push(2); m /= 2; }
  for (int q = 3; m > 1; q += 2)
    while (m % q == 0) { push(q); m /= q; }
  p.by_n = make_gen_div(n);
  p.by_nl = make_gen_div(p.nl);
  return p;
}

// Dynamic LDS of a pass: the N twiddles (FP64, of a length whose outputs are
// formed directly in the lines' precision) and the line buffer (padded stride
// N + 1; two of them for the latter).
template <typename T>
inline size_t gen_smem(int n) {
  const GenPlan p = make_gen_plan(n);
  return size_t(p.direct ? 2 : 1) * p.nl * (n + 1) * sizeof(c2<T>) +
         size_t(n) * (p.direct ? sizeof(c2<T>) : sizeof(double2));
}

// x <- DFT_P(x), P odd: with s_q = x_q + x_{P-q}, d_q = x_q - x_{P-q},
// X_{r, P-r} = x_0 + sum_q cos(2 pi q r / P) s_q +- i sgn sum_q sin(..) d_q.
template <typename T, int P>
__device__ __forceinline__ void dft_odd(c2<T>* x, T sgn) {
  constexpr int H = (P - 1) / 2;
  c2<T> s[H], d[H];
#pragma unroll
  for (int q = 1; q <= H; q++) {
    s[q - 1] = cadd<T>(x[q], x[P - q]);
    d[q - 1] = csub<T>(x[q], x[P - q]);
  }
  const c2<T> x0 = x[0];
#pragma unroll
  for (int q = 0; q < H; q++) x[0] = cadd<T>(x[0], s[q]);
#pragma unroll
  for (int r = 1; r <= H; r++) {
    c2<T> u = x0, v = mk<T>(T(0), T(0));
#pragma unroll
    for (int q = 1; q <= H; q++) {
      const T c = T(cx_series(cx_turn(q * r, P), false));
      const T w = T(cx_series(cx_turn(q * r, P), true));
      u.x += c * s[q - 1].x;
      u.y += c * s[q - 1].y;
      v.x += w * d[q - 1].x;
      v.y += w * d[q - 1].y;
    }
    const c2<T> iv = mk<T>(-sgn * v.y, sgn * v.x);
    x[r] = cadd<T>(u, iv);
    x[P - r] = csub<T>(u, iv);
  }
}

// Stage s of radix P over the buffer `a`, in place.
template <typename T, int P>
__device__ __forceinline__ void gen_stage(c2<T>* a, const double2* W, const GenPlan& pl, int s,
                                          int Ns, int nl, double sgn) {
  constexpr int NB = (GEN_ELEMS / P + FFT_THREADS - 1) / FFT_THREADS;
  const int N = pl.n, LS = N + 1, Np = N / P, total = nl * Np;
  const int tstep = N / (Ns * P);
  c2<T> x[NB][P];
  int d[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const int o = threadIdx.x + b * FFT_THREADS;
    if (o >= total) continue;
    const int line = pl.by_np[s].div(o), j = o - line * Np;
    const int jq = pl.by_ns[s].div(j), k = j - jq * Ns;
    const c2<T>* src = a + line * LS + j;
    d[b] = line * LS + jq * Ns * P + k;
    double2 y[P];
#pragma unroll
    for (int q = 0; q < P; q++) {
      const c2<T> v = src[q * Np];
      y[q] = dmk(v.x, v.y);
      if (q > 0) y[q] = dmul(y[q], W[q * k * tstep]);
    }
    if constexpr (P % 2 == 0) dft_reg<double, P>(y, sgn);
    else dft_odd<double, P>(y, sgn);
#pragma unroll
    for (int q = 0; q < P; q++) x[b][q] = mk<T>(T(y[q].x), T(y[q].y));
  }
  __syncthreads();
#pragma unroll
  for (int b = 0; b < NB; b++) {
    if (int(threadIdx.x) + b * FFT_THREADS >= total) continue;
#pragma unroll
    for (int r = 0; r < P; r++) a[d[b] + r * Ns] = x[b][r];
  }
  __syncthreads();
}

// The nl lines of a (line stride N + 1) are transformed; returns the buffer
// (a, or b of the direct lengths) holding the result.  Ends with a barrier.
template <typename T>
__device__ __forceinline__ c2<T>* lds_fft_gen(c2<T>* a, c2<T>* b, const void* tw,
                                              const GenPlan& P, int nl, int sign) {
  const int N = P.n, LS = N + 1;
  int Ns = 1;
  if (!P.direct) {
    const double2* W = static_cast<const double2*>(tw);
    for (int s = 0; s < P.nst; s++) {
      switch (P.radix[s]) {
        case 2: gen_stage<T, 2>(a, W, P, s, Ns, nl, sign); break;
        case 3: gen_stage<T, 3>(a, W, P, s, Ns, nl, sign); break;
        case 4: gen_stage<T, 4>(a, W, P, s, Ns, nl, sign); break;
        case 5: gen_stage<T, 5>(a, W, P, s, Ns, nl, sign); break;
        default: gen_stage<T, 7>(a, W, P, s, Ns, nl, sign); break;
      }
      Ns *= P.radix[s];
    }
    return a;
  }
  const c2<T>* W = static_cast<const c2<T>*>(tw);
  const int total = nl * N;
  for (int s = 0; s < P.nst; s++) {
    const int p = P.radix[s];
    const int Np = N / p;
    const int tstep = N / (Ns * p);
    for (int o = threadIdx.x; o < total; o += FFT_THREADS) {
      const int line = P.by_n.div(o), rem = o - line * N;
      const int r = P.by_np[s].div(rem), j = rem - r * Np;
      const int jq = P.by_ns[s].div(j), k = j - jq * Ns;
      int be = k * tstep + r * Np;
      if (be >= N) be -= N;
      const c2<T>* src = a + line * LS + j;
      c2<T> acc = mk<T>(T(0), T(0));
      int e = 0;
      for (int q = 0; q < p; q++) {
        acc = cadd<T>(acc, cmul<T>(src[q * Np], W[e]));
        e += be;
        if (e >= N) e -= N;
      }
      b[line * LS + jq * Ns * p + k + r * Ns] = acc;
    }
    __syncthreads();
    c2<T>* t = a;
    a = b;
    b = t;
    Ns *= p;
  }
  return a;
}

// LDS of a pass, and its twiddles copied there from the table `tw`.
template <typename T>
struct GenSmem {
  c2<T>* a;
  c2<T>* b;
  void* W;
  __device__ explicit GenSmem(const GenPlan& P) {
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    W = smem_raw;
    a = reinterpret_cast<c2<T>*>(smem_raw +
                                 P.n * (P.direct ? sizeof(c2<T>) : sizeof(double2)));
    b = a + P.nl * (P.n + 1);
  }
  __device__ __forceinline__ void fill(const GenPlan& P, const void* tw) const {
    if (P.direct) {
      for (int m = threadIdx.x; m < P.n; m += FFT_THREADS)
        static_cast<c2<T>*>(W)[m] = static_cast<const c2<T>*>(tw)[m];
    } else {
      for (int m = threadIdx.x; m < P.n; m += FFT_THREADS)
        static_cast<double2*>(W)[m] = static_cast<const double2*>(tw)[m];
    }
  }
};

// Quotient and remainder by `d` of x0 + l, from those of x0, for small l.
struct GenSplit {
  unsigned q0, r0, d;
  __device__ GenSplit(long long x0, long long div)
      : q0(unsigned(x0) / unsigned(div)), r0(unsigned(x0) % unsigned(div)), d(unsigned(div)) {}
  __device__ __forceinline__ void at(int l, int& q, int& r) const {
    unsigned qq = q0, rr = r0 + unsigned(l);
    while (rr >= d) { rr -= d; qq++; }
    q = int(qq);
    r = int(rr);
  }
};

// z pass (contiguous lines, line index = i n1 + j) with a loader.
template <typename T, class Loader>
__device__ __forceinline__ void fft_z_block_gen(c2<T>* __restrict__ data, const Loader& load,
                                const void* __restrict__ tw, int n1, long long nlines,
                                int sign, const Prune& pr, const GenPlan& P,
                                long long blk) {
  const int N = P.n;
  GenSmem<T> sm(P);
  const long long line0 = blk * P.nl;
  if (line0 >= nlines) return;
  const int nl = int(min((long long)P.nl, nlines - line0)), total = nl * N;
  const GenSplit ij(line0, n1);
  if (pr.on) {
    bool any = false;
    for (int l = 0; l < nl && !any; l++) {
      int i, j;
      ij.at(l, i, j);
      any = pr.p1(i, j);
    }
    if (!any) return;
  }
  sm.fill(P, tw);
  // Threads past the end repeat the last element (no branch, so the loads
  // stay in flight together).
  c2<T> v[GEN_MAXE];
#pragma unroll
  for (int e = 0; e < GEN_MAXE; e++) {
    const int idx = min(int(threadIdx.x) + e * FFT_THREADS, total - 1);
    const int l = P.by_n.div(idx);
    int i, j;
    ij.at(l, i, j);
    v[e] = load(line0 * N + idx, i, j, idx - l * N);
    if (HeavyLoader<Loader>::value && e % 4 == 3) __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int e = 0; e < GEN_MAXE; e++) {
    const int idx = threadIdx.x + e * FFT_THREADS;
    if (idx < total) sm.a[idx + P.by_n.div(idx)] = v[e];   // line stride N + 1
  }
  __syncthreads();
  const c2<T>* R = lds_fft_gen<T>(sm.a, sm.b, sm.W, P, nl, sign);
#pragma unroll
  for (int e = 0; e < GEN_MAXE; e++) {
    const int idx = threadIdx.x + e * FFT_THREADS;
    if (idx < total) st_mesh<T>(data + line0 * N + idx, R[idx + P.by_n.div(idx)]);
  }
}

template <typename T, class Loader>
__global__ void __launch_bounds__(FFT_THREADS)
fft_pass_z_gen(c2<T>* __restrict__ data, Loader load, const void* __restrict__ tw,
               int n1, long long nlines, int sign, Prune pr, GenPlan P) {
  fft_z_block_gen<T>(data, load, tw, n1, nlines, sign, pr, P, blockIdx.x);
}

template <typename T, class BatchLoader>
__global__ void __launch_bounds__(FFT_THREADS)
fft_pass_z_batch_gen(c2<T>* __restrict__ base, long long fstride, BatchLoader load,
                     const void* __restrict__ tw, int n1, long long nlines, int sign,
                     Prune pr, const double* __restrict__ kcut2,
                     const int2* __restrict__ work, GenPlan P) {
  const int2 wk = work[blockIdx.x];
  Prune p = pr;
  p.kcut2 = kcut2[wk.x];
  fft_z_block_gen<T>(base + wk.x * fstride, load.field(wk.x), tw, n1, nlines, sign, p,
                     P, wk.y);
}

// Strided pass (line `id` starts at (id / inner) outer_stride + id % inner,
// element stride S) with the pruning modes of fft_strided_block.
template <typename T>
__device__ __forceinline__ void fft_strided_block_gen(
    c2<T>* __restrict__ data, const void* __restrict__ tw, long long S,
    long long outer_stride, long long inner, long long nlines, int sign, const Prune& pr,
    int prune_mode, const GenPlan& P, long long blk) {
  const int N = P.n, LS = N + 1;
  GenSmem<T> sm(P);
  const long long id0 = blk * P.nl;
  if (id0 >= nlines) return;
  const int nl = int(min((long long)P.nl, nlines - id0)), total = nl * N;
  const GenSplit sc(id0, inner);
  if (pr.on && prune_mode != 2) {
    bool any = false;
    for (int l = 0; l < nl && !any; l++) {
      int slice, col;
      sc.at(l, slice, col);
      any = pr.p2(prune_mode == 1 ? slice : col);
    }
    if (!any) return;
  }
  sm.fill(P, tw);
  // Element (n, l): consecutive threads take consecutive lines (nl of them,
  // which is P.nl but in the last block).
  const bool whole = nl == P.nl;
  auto split = [&](int idx, int& n, int& l) {
    n = whole ? P.by_nl.div(idx) : idx / nl;
    l = idx - n * nl;
  };
  c2<T>* at[GEN_MAXE];
  c2<T> v[GEN_MAXE];
  bool out[GEN_MAXE];
#pragma unroll
  for (int e = 0; e < GEN_MAXE; e++) {
    const int idx = min(int(threadIdx.x) + e * FFT_THREADS, total - 1);
    int n, l, slice, col;
    split(idx, n, l);
    sc.at(l, slice, col);
    at[e] = data + (long long)slice * outer_stride + col + (long long)n * S;
    bool need = true;
    out[e] = true;
    if (pr.on) {
      if (prune_mode == 1) {
        out[e] = pr.p2(slice);
        need = out[e] && pr.p1(slice, n);
      } else if (prune_mode == 2) {
        need = pr.p2(n);
      } else {
        out[e] = pr.p2(col);
        need = pr.p1(col, n);
      }
    }
    v[e] = need ? ld_mesh<T>(at[e]) : mk<T>(T(0), T(0));
  }
#pragma unroll
  for (int e = 0; e < GEN_MAXE; e++) {
    const int idx = threadIdx.x + e * FFT_THREADS;
    int n, l;
    split(idx, n, l);
    if (idx < total) sm.a[l * LS + n] = v[e];
  }
  __syncthreads();
  const c2<T>* R = lds_fft_gen<T>(sm.a, sm.b, sm.W, P, nl, sign);
#pragma unroll
  for (int e = 0; e < GEN_MAXE; e++) {
    const int idx = threadIdx.x + e * FFT_THREADS;
    int n, l;
    split(idx, n, l);
    if (idx < total && out[e]) st_mesh<T>(at[e], R[l * LS + n]);
  }
}

template <typename T>
__global__ void __launch_bounds__(FFT_THREADS)
fft_pass_strided_gen(c2<T>* __restrict__ data, const void* __restrict__ tw, long long S,
                     long long outer_stride, long long inner, long long nlines, int sign,
                     Prune pr, int prune_mode, GenPlan P) {
  fft_strided_block_gen<T>(data, tw, S, outer_stride, inner, nlines, sign, pr, prune_mode, P,
                           blockIdx.x);
}

template <typename T>
__global__ void __launch_bounds__(FFT_THREADS)
fft_pass_strided_batch_gen(c2<T>* __restrict__ base, long long fstride,
                           const void* __restrict__ tw, long long S, long long outer_stride,
                           long long inner, long long nlines, int sign, Prune pr,
                           const double* __restrict__ kcut2, const int2* __restrict__ work,
                           int prune_mode, GenPlan P) {
  const int2 wk = work[blockIdx.x];
  Prune p = pr;
  p.kcut2 = kcut2[wk.x];
  fft_strided_block_gen<T>(base + wk.x * fstride, tw, S, outer_stride, inner, nlines, sign, p,
                           prune_mode, P, wk.y);
}

// First pass of the x-first order: lines along x (element stride n1 n2,
// line id = j n2 + k) with a loader load(g, i, j, k); blocks with no line
// where P1(k, j) are skipped.
template <typename T, class Loader>
__device__ __forceinline__ void fft_x_load_block_gen(c2<T>* __restrict__ data,
                                     const Loader& load,
                                     const void* __restrict__ tw, int n1, int n2,
                                     const Prune& pr, const GenPlan& P, long long blk) {
  const int N = P.n, LS = N + 1;
  GenSmem<T> sm(P);
  const long long S = (long long)n1 * n2;
  const long long id0 = blk * P.nl;
  if (id0 >= S) return;
  const int nl = int(min((long long)P.nl, S - id0)), total = nl * N;
  const GenSplit jk(id0, n2);
  if (pr.on) {
    bool any = false;
    for (int l = 0; l < nl && !any; l++) {
      int j, k;
      jk.at(l, j, k);
      any = pr.p1(k, j);
    }
    if (!any) return;
  }
  sm.fill(P, tw);
  const bool whole = nl == P.nl;
  auto split = [&](int idx, int& n, int& l) {
    n = whole ? P.by_nl.div(idx) : idx / nl;
    l = idx - n * nl;
  };
#pragma unroll
  for (int e = 0; e < GEN_MAXE; e++) {
    const int idx = threadIdx.x + e * FFT_THREADS;
    if (idx >= total) continue;
    int n, l, j, k;
    split(idx, n, l);
    jk.at(l, j, k);
    sm.a[l * LS + n] = load(id0 + l + (long long)n * S, n, j, k);
  }
  __syncthreads();
  const c2<T>* R = lds_fft_gen<T>(sm.a, sm.b, sm.W, P, nl, +1);
#pragma unroll
  for (int e = 0; e < GEN_MAXE; e++) {
    const int idx = threadIdx.x + e * FFT_THREADS;
    int n, l;
    split(idx, n, l);
    if (idx < total) st_mesh<T>(data + id0 + l + (long long)n * S, R[l * LS + n]);
  }
}

template <typename T, class BatchLoader>
__global__ void __launch_bounds__(FFT_THREADS)
fft_pass_x_load_batch_gen(c2<T>* __restrict__ base, long long fstride, BatchLoader load,
                          const void* __restrict__ tw, int n1, int n2, Prune pr,
                          const double* __restrict__ kcut2, const int2* __restrict__ work,
                          GenPlan P) {
  const int2 wk = work[blockIdx.x];
  Prune p = pr;
  p.kcut2 = kcut2[wk.x];
  fft_x_load_block_gen<T>(base + wk.x * fstride, load.field(wk.x), tw, n1, n2, p, P,
                          wk.y);
}

}  // namespace trvg

// engine_fft.hpp -- launches of the mesh transforms: full 3-D transforms
// with fused first-pass loaders, batched transforms over work lists, and
// the shell slabs of the estimators.  Included by the two translation units
// that instantiate them (engine_fft64.hip, engine_fft32.hip).
#pragma once

#include <algorithm>
#include <map>
#include <tuple>

#include "batch_kernels.hpp"
#include "diff_kernels.hpp"
#include "engine.hpp"
#include "prune_lists.hpp"

namespace trvg {

// ---------------------------------------------------------------------------
// FFT
// ---------------------------------------------------------------------------

template <typename T>
static const c2<T>* twiddles(int n, int sign);

// Twiddles of a transform in context ctx: borrowed tables where the context
// has them, else the engine's cache.
template <typename T>
static const c2<T>* ctx_twiddles(const Context& ctx, int n, int sign) {
  int lg = 0;
  while ((1 << lg) < n) lg++;
  const void* b = (lg < 11 && (1 << lg) == n) ? ctx.tw[sign > 0 ? 1 : 0][lg] : nullptr;
  return b ? static_cast<const c2<T>*>(b) : twiddles<T>(n, sign);
}

template <typename T>
static const c2<T>* twiddles(int n, int sign) {
  static std::mutex mu;
  static std::map<std::tuple<int, int, int>, c2<T>*> cache;
  int dev = 0;
  TRVG_HIP(hipGetDevice(&dev));
  auto key = std::make_tuple(dev, n, sign);
  std::lock_guard<std::mutex> lk(mu);
  auto it = cache.find(key);
  if (it != cache.end()) return it->second;
  std::vector<c2<T>> h(n);
  for (int m = 0; m < n; m++) {
    double a = 2. * M_PI * double(m) / double(n);
    h[m] = mk<T>(T(std::cos(a)), T(sign * std::sin(a)));
  }
  c2<T>* d = nullptr;
  TRVG_HIP(hipMalloc(&d, n * sizeof(c2<T>)));
  TRVG_HIP(hipMemcpy(d, h.data(), n * sizeof(c2<T>), hipMemcpyHostToDevice));
  cache[key] = d;
  return d;
}


// Dynamic LDS above the default 64 KiB needs the kernel's attribute raised.
template <class K>
static void raise_lds(K kernel, size_t bytes) {
  if (bytes > 64 * 1024)
    TRVG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes)));
}

template <typename T, int LOGN, class Loader>
static void launch_z(Context& ctx, c2<T>* data, const Loader& load, int sign,
                     double read_bytes, double write_bytes, const Prune& pr) {
  constexpr int N = 1 << LOGN;
  const long long nlines = ctx.g.nmesh / N;
  const c2<T>* tw = ctx_twiddles<T>(ctx, N, sign);
  ProfScope ps(ctx, sizeof(T) == 8 ? KC_FFT_Z64 : KC_FFT_Z, read_bytes + write_bytes);
  hipLaunchKernelGGL((fft_pass_z<T, LOGN, Loader>),
                     dim3(unsigned((nlines + z_lines(N) - 1) / z_lines(N))), dim3(FFT_THREADS),
                     (z_smem<T, LOGN>()), ctx.stream, data, load, tw, ctx.g.n[1], nlines, sign,
                     pr);
  TRVG_LAUNCH_CHECK();
}

template <typename T, int LOGN>
static void launch_strided(Context& ctx, c2<T>* data, long long S,
                           long long outer_stride, long long inner, int sign,
                           const Prune& pr, int prune_mode, double bytes) {
  constexpr int NL = strided_lines<T, LOGN>();
  const long long nlines = ctx.g.nmesh >> LOGN;
  const c2<T>* tw = ctx_twiddles<T>(ctx, 1 << LOGN, sign);
  ProfScope ps(ctx, sizeof(T) == 8 ? KC_FFT_STRIDED64 : KC_FFT_STRIDED, bytes);
  auto kern = fft_pass_strided<T, LOGN>;
  raise_lds(kern, strided_smem<T, LOGN>());
  hipLaunchKernelGGL(kern, dim3(unsigned((nlines + NL - 1) / NL)),
                     dim3(strided_threads<T, LOGN>()), (strided_smem<T, LOGN>()), ctx.stream,
                     data, tw, S, outer_stride, inner, nlines, sign, pr, prune_mode);
  TRVG_LAUNCH_CHECK();
}

static int ilog2(int n) {
  int l = 0;
  while ((1 << l) < n) l++;
  return l;
}

#define TRVG_LOGN_SWITCH(lg, CALL)                               \
  switch (lg) {                                                  \
    case 3: { constexpr int LG = 3; CALL; } break;               \
    case 4: { constexpr int LG = 4; CALL; } break;               \
    case 5: { constexpr int LG = 5; CALL; } break;               \
    case 6: { constexpr int LG = 6; CALL; } break;               \
    case 7: { constexpr int LG = 7; CALL; } break;               \
    case 8: { constexpr int LG = 8; CALL; } break;               \
    case 9: { constexpr int LG = 9; CALL; } break;               \
    case 10: { constexpr int LG = 10; CALL; } break;             \
    default: throw Error(TRVG_ERR_PARAM, "Unsupported FFT size."); \
  }

// Axes of power-of-two length up to 1024 take the compile-time passes of
// fft.hpp; other (even) lengths the mixed-radix passes of fft_gen.hpp.
static bool fast_axis(int n) { return n >= 8 && n <= 1024 && (n & (n - 1)) == 0; }
// Lines per workgroup of the z pass and of the strided passes (work lists).
static int lines_z(int n) { return fast_axis(n) ? z_lines(n) : gen_lines_per_block(n); }
template <typename T>
static int lines_strided(int n) {
  if (fast_axis(n)) {
    TRVG_LOGN_SWITCH(ilog2(n), return (strided_lines<T, LG>()));
  }
  return gen_lines_per_block(n);
}
static long long blocks_of(long long nlines, int nl) { return (nlines + nl - 1) / nl; }

// Twiddles of a mixed-radix pass: FP64 but where outputs are formed directly.
template <typename T>
static const void* gen_twiddles(const Context& ctx, const GenPlan& P, int sign) {
  if (P.direct) return ctx_twiddles<T>(ctx, P.n, sign);
  return ctx_twiddles<double>(ctx, P.n, sign);
}

template <typename T, class Loader>
static void launch_z_gen(Context& ctx, c2<T>* data, const Loader& load, int sign,
                         double bytes, const Prune& pr) {
  const int N = ctx.g.n[2];
  const GenPlan P = make_gen_plan(N);
  const long long nlines = (long long)ctx.g.n[0] * ctx.g.n[1];
  const size_t smem = gen_smem<T>(N);
  auto kern = fft_pass_z_gen<T, Loader>;
  raise_lds(kern, smem);
  ProfScope ps(ctx, sizeof(T) == 8 ? KC_FFT_Z64 : KC_FFT_Z, bytes);
  hipLaunchKernelGGL(kern, dim3(unsigned(blocks_of(nlines, P.nl))), dim3(FFT_THREADS), smem,
                     ctx.stream, data, load, gen_twiddles<T>(ctx, P, sign), ctx.g.n[1],
                     nlines, sign, pr, P);
  TRVG_LAUNCH_CHECK();
}

template <typename T>
static void launch_strided_gen(Context& ctx, c2<T>* data, int N, long long S,
                               long long outer_stride, long long inner, int sign,
                               const Prune& pr, int prune_mode, double bytes) {
  const GenPlan P = make_gen_plan(N);
  const long long nlines = ctx.g.nmesh / N;
  const size_t smem = gen_smem<T>(N);
  auto kern = fft_pass_strided_gen<T>;
  raise_lds(kern, smem);
  ProfScope ps(ctx, sizeof(T) == 8 ? KC_FFT_STRIDED64 : KC_FFT_STRIDED, bytes);
  hipLaunchKernelGGL(kern, dim3(unsigned(blocks_of(nlines, P.nl))), dim3(FFT_THREADS), smem,
                     ctx.stream, data, gen_twiddles<T>(ctx, P, sign), S, outer_stride, inner,
                     nlines, sign, pr, prune_mode, P);
  TRVG_LAUNCH_CHECK();
}

template <typename T, class BatchLoader>
static void launch_z_batch_gen(Context& ctx, c2<T>* base, const BatchLoader& load, int sign,
                               const Prune& pr, const double* kcut2, const int2* work,
                               int nwork, double bytes) {
  const int N = ctx.g.n[2];
  const GenPlan P = make_gen_plan(N);
  const long long nlines = (long long)ctx.g.n[0] * ctx.g.n[1];
  const size_t smem = gen_smem<T>(N);
  auto kern = fft_pass_z_batch_gen<T, BatchLoader>;
  raise_lds(kern, smem);
  ProfScope ps(ctx, sizeof(T) == 8 ? KC_FFT_Z64 : KC_FFT_Z, bytes);
  hipLaunchKernelGGL(kern, dim3(unsigned(nwork)), dim3(FFT_THREADS), smem, ctx.stream, base,
                     ctx.g.nmesh, load, gen_twiddles<T>(ctx, P, sign), ctx.g.n[1], nlines,
                     sign, pr, kcut2, work, P);
  TRVG_LAUNCH_CHECK();
}

template <typename T>
static void launch_strided_batch_gen(Context& ctx, c2<T>* base, int N, long long S,
                                     long long outer_stride, long long inner, int sign,
                                     const Prune& pr, const double* kcut2, const int2* work,
                                     int nwork, int prune_mode, double bytes) {
  const GenPlan P = make_gen_plan(N);
  const long long nlines = ctx.g.nmesh / N;
  const size_t smem = gen_smem<T>(N);
  auto kern = fft_pass_strided_batch_gen<T>;
  raise_lds(kern, smem);
  ProfScope ps(ctx, sizeof(T) == 8 ? KC_FFT_STRIDED64 : KC_FFT_STRIDED, bytes);
  hipLaunchKernelGGL(kern, dim3(unsigned(nwork)), dim3(FFT_THREADS), smem, ctx.stream, base,
                     ctx.g.nmesh, gen_twiddles<T>(ctx, P, sign), S, outer_stride, inner,
                     nlines, sign, pr, kcut2, work, prune_mode, P);
  TRVG_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// Batched shell transforms: one launch per pass for a whole slab of bins,
// over only the blocks whose lines lie in each bin's band.
// ---------------------------------------------------------------------------

// Work lists of one geometry, pass shape and radius (prune_lists.hpp), built
// once.
static const PruneLists& prune_lists(const Geom& g, double kcut2, int nl_z,
                                     int nl_y) {
  static std::mutex mu;
  static std::map<std::vector<double>, std::unique_ptr<PruneLists>> cache;
  std::vector<double> key = {double(g.n[0]), double(g.n[1]), double(g.n[2]),
                             g.dk[0], g.dk[1], kcut2, double(nl_z), double(nl_y)};
  std::lock_guard<std::mutex> lk(mu);
  auto it = cache.find(key);
  if (it != cache.end()) return *it->second;
  auto pl = std::make_unique<PruneLists>(make_prune_lists(g.n, g.dk, kcut2, nl_z, nl_y));
  return *(cache[key] = std::move(pl));
}

template <typename T, int LOGN, class BatchLoader>
static void launch_z_batch(Context& ctx, c2<T>* base, const BatchLoader& load,
                           int sign, const Prune& pr, const double* kcut2,
                           const int2* work, int nwork, double bytes) {
  constexpr int N = 1 << LOGN;
  const c2<T>* tw = ctx_twiddles<T>(ctx, N, sign);
  ProfScope ps(ctx, sizeof(T) == 8 ? KC_FFT_Z64 : KC_FFT_Z, bytes);
  hipLaunchKernelGGL((fft_pass_z_batch<T, LOGN, BatchLoader>), dim3(unsigned(nwork)),
                     dim3(FFT_THREADS), (z_smem<T, LOGN>()), ctx.stream, base, ctx.g.nmesh,
                     load, tw, ctx.g.n[1], ctx.g.nmesh / N, sign, pr, kcut2, work);
  TRVG_LAUNCH_CHECK();
}

template <typename T, int LOGN>
static void launch_strided_batch(Context& ctx, c2<T>* base, long long S,
                                 long long outer_stride, long long inner,
                                 int sign, const Prune& pr, const double* kcut2,
                                 const int2* work, int nwork, int prune_mode,
                                 double bytes) {
  const c2<T>* tw = ctx_twiddles<T>(ctx, 1 << LOGN, sign);
  ProfScope ps(ctx, sizeof(T) == 8 ? KC_FFT_STRIDED64 : KC_FFT_STRIDED, bytes);
  auto kern = fft_pass_strided_batch<T, LOGN>;
  raise_lds(kern, strided_smem<T, LOGN>());
  hipLaunchKernelGGL(kern, dim3(unsigned(nwork)), dim3(strided_threads<T, LOGN>()),
                     (strided_smem<T, LOGN>()), ctx.stream, base, ctx.g.nmesh, tw, S,
                     outer_stride, inner, ctx.g.nmesh >> LOGN, sign, pr, kcut2, work,
                     prune_mode);
  TRVG_LAUNCH_CHECK();
}

// Transform of several fields in one launch per pass: field f of the work
// lists lives at base + f * nmesh and loads through load.field(f); with
// `prune`, kcut2[f] is field f's pruning radius and the lists hold only the
// blocks that radius needs (z and y passes).
template <typename T, class BatchLoader>
void fft3d_batch(Context& ctx, c2<T>* base, const BatchLoader& load, int sign,
                 bool prune, const double* kcut2, const int2* wz, int nz,
                 const int2* wy, int ny, const int2* wx, int nx) {
  const Geom& g = ctx.g;
  Prune pr{};
  pr.on = prune ? 1 : 0;
  pr.dk0 = g.dk[0];
  pr.dk1 = g.dk[1];
  pr.n0 = g.n[0];
  pr.n1 = g.n[1];
  // Bytes of a listed block of an axis of n points with nl lines each.
  auto blk = [](int n, int nl) { return double(nl) * n * sizeof(c2<T>); };
  const double bz = 2. * nz * blk(g.n[2], lines_z(g.n[2]));
  const double by = 2. * ny * blk(g.n[1], lines_strided<T>(g.n[1]));
  const double bx = 2. * nx * blk(g.n[0], lines_strided<T>(g.n[0]));
  if (nz > 0) {
    if (fast_axis(g.n[2])) {
      TRVG_LOGN_SWITCH(ilog2(g.n[2]), (launch_z_batch<T, LG>(
          ctx, base, load, sign, pr, kcut2, wz, nz, bz)));
    } else {
      launch_z_batch_gen<T>(ctx, base, load, sign, pr, kcut2, wz, nz, bz);
    }
  }
  if (ny > 0) {
    if (fast_axis(g.n[1])) {
      TRVG_LOGN_SWITCH(ilog2(g.n[1]), (launch_strided_batch<T, LG>(
          ctx, base, g.n[2], (long long)g.n[1] * g.n[2], g.n[2], sign, pr, kcut2, wy,
          ny, 1, by)));
    } else {
      launch_strided_batch_gen<T>(ctx, base, g.n[1], g.n[2], (long long)g.n[1] * g.n[2],
                                  g.n[2], sign, pr, kcut2, wy, ny, 1, by);
    }
  }
  if (nx > 0) {
    if (fast_axis(g.n[0])) {
      TRVG_LOGN_SWITCH(ilog2(g.n[0]), (launch_strided_batch<T, LG>(
          ctx, base, (long long)g.n[1] * g.n[2], 0, (long long)g.n[1] * g.n[2], sign,
          pr, kcut2, wx, nx, 2, bx)));
    } else {
      launch_strided_batch_gen<T>(ctx, base, g.n[0], (long long)g.n[1] * g.n[2], 0,
                                  (long long)g.n[1] * g.n[2], sign, pr, kcut2, wx, nx, 2,
                                  bx);
    }
  }
}

// Every block of nf meshes, per pass.
template <typename T>
void full_work(const Geom& g, int nf, std::vector<int2>& wz, std::vector<int2>& wy,
               std::vector<int2>& wx) {
  auto fill = [&](int axis, int nl, std::vector<int2>& w) {
    w.clear();
    const long long nb = blocks_of(g.nmesh / g.n[axis], nl);
    for (int f = 0; f < nf; f++)
      for (long long b = 0; b < nb; b++) w.push_back(make_int2(f, int(b)));
  };
  fill(2, lines_z(g.n[2]), wz);
  fill(1, lines_strided<T>(g.n[1]), wy);
  fill(0, lines_strided<T>(g.n[0]), wx);
}

// Work lists of a shell slab transform over `ngroups` groups of all
// `nbins` bins: per group nt transforms (nbins, or (nbins + 1) / 2 when
// packed, two real bins per transform), transform f = group * nt + t.
// Returns the bins' bands (two per transform when packed, padded with an
// empty band), each transform's pruning radius (+inf when the band covers
// the whole plane), and the z / y / x blocks.
template <typename T>
void shell_slab_work(const Geom& g, const trvg_binning& kb, int nbins,
                     int ngroups, bool packed, std::vector<ShellBand>& bands,
                     std::vector<double>& kcut2, std::vector<int2>& wz,
                     std::vector<int2>& wy, std::vector<int2>& wx) {
  const int nl_z = lines_z(g.n[2]), nl_y = lines_strided<T>(g.n[1]);
  const long long nblk = blocks_of((long long)g.n[1] * g.n[2], lines_strided<T>(g.n[0]));
  const int per = packed ? 2 : 1;
  const int nt = (nbins + per - 1) / per;
  bands.assign((size_t)nt * per, ShellBand{HUGE_VAL, HUGE_VAL});
  std::vector<double> kc(nt, 0.);
  for (int q = 0; q < nbins; q++) {
    bands[q] = shell_band(kb.bin_edges[q], kb.bin_edges[q + 1]);
    Prune pq = make_prune(g, kb.bin_edges[q + 1]);
    kc[q / per] = std::max(kc[q / per], pq.on ? pq.kcut2 : HUGE_VAL);
  }
  std::vector<const PruneLists*> pls(nt);
  for (int t = 0; t < nt; t++) pls[t] = &prune_lists(g, kc[t], nl_z, nl_y);
  kcut2.clear(); wz.clear(); wy.clear(); wx.clear();
  for (int gi = 0; gi < ngroups; gi++)
    for (int t = 0; t < nt; t++) {
      const int f = gi * nt + t;
      kcut2.push_back(kc[t]);
      for (int w : pls[t]->zblocks) wz.push_back(make_int2(f, w));
      for (int w : pls[t]->yblocks) wy.push_back(make_int2(f, w));
      for (long long w = 0; w < nblk; w++) wx.push_back(make_int2(f, int(w)));
    }
}

// ---------------------------------------------------------------------------
// Shell transforms, x-first: the x pass carries the shell loader (lines
// along x at fixed (k_y, k_z), pruned on k_y^2 + k_z^2), the y pass is
// pruned on k_z, and the last pass runs along the contiguous z lines, so
// the full-size output of every field is written in whole 16 KiB blocks
// rather than as short strided segments.
// ---------------------------------------------------------------------------

// Prune over the (z, y) axes: P2(k) tests k_z, P1(k, j) tests (k_z, k_y).
static Prune prune_zy(const Geom& g) {
  Prune pr{};
  pr.on = 1;
  pr.dk0 = g.dk[2];
  pr.dk1 = g.dk[1];
  pr.n0 = g.n[2];
  pr.n1 = g.n[1];
  return pr;
}

static const PruneListsXF& prune_lists_xfirst(const Geom& g, double kcut2, int nl_x,
                                              int nl_y) {
  static std::mutex mu;
  static std::map<std::vector<double>, std::unique_ptr<PruneListsXF>> cache;
  std::vector<double> key = {double(g.n[0]), double(g.n[1]), double(g.n[2]),
                             g.dk[1], g.dk[2], kcut2, double(nl_x), double(nl_y)};
  std::lock_guard<std::mutex> lk(mu);
  auto it = cache.find(key);
  if (it != cache.end()) return *it->second;
  auto pl =
      std::make_unique<PruneListsXF>(make_prune_lists_xfirst(g.n, g.dk, kcut2, nl_x, nl_y));
  return *(cache[key] = std::move(pl));
}

template <typename T, int LOGN, class BatchLoader>
static void launch_x_load_batch(Context& ctx, c2<T>* base, const BatchLoader& load,
                                const Prune& pr, const double* kcut2, const int2* work,
                                int nwork, double bytes) {
  const c2<T>* tw = ctx_twiddles<T>(ctx, 1 << LOGN, +1);
  ProfScope ps(ctx, sizeof(T) == 8 ? KC_FFT_STRIDED64 : KC_FFT_STRIDED, bytes);
  auto kern = fft_pass_x_load_batch<T, LOGN, BatchLoader>;
  raise_lds(kern, strided_smem<T, LOGN>());
  hipLaunchKernelGGL(kern, dim3(unsigned(nwork)), dim3(strided_threads<T, LOGN>()),
                     (strided_smem<T, LOGN>()), ctx.stream, base, ctx.g.nmesh, load, tw,
                     ctx.g.n[1], ctx.g.n[2], +1, pr, kcut2, work);
  TRVG_LAUNCH_CHECK();
}

template <typename T, class BatchLoader>
static void launch_x_load_batch_gen(Context& ctx, c2<T>* base, const BatchLoader& load,
                                    const Prune& pr, const double* kcut2, const int2* work,
                                    int nwork, double bytes) {
  const int N = ctx.g.n[0];
  const GenPlan P = make_gen_plan(N);
  const size_t smem = gen_smem<T>(N);
  auto kern = fft_pass_x_load_batch_gen<T, BatchLoader>;
  raise_lds(kern, smem);
  ProfScope ps(ctx, sizeof(T) == 8 ? KC_FFT_STRIDED64 : KC_FFT_STRIDED, bytes);
  hipLaunchKernelGGL(kern, dim3(unsigned(nwork)), dim3(FFT_THREADS), smem, ctx.stream, base,
                     ctx.g.nmesh, load, gen_twiddles<T>(ctx, P, +1), ctx.g.n[1], ctx.g.n[2],
                     pr, kcut2, work, P);
  TRVG_LAUNCH_CHECK();
}

template <typename T>
static void xfirst_yz(Context& ctx, c2<T>* base, const double* kcut2, const int2* wy, int ny,
                      const int2* wz, int nz, double by, double bz);

// The three passes of a batched x-first transform: field f of the work
// lists lives at base + f * nmesh, loads through load.field(f) and is pruned
// with radius kcut2[f] (+inf: no pruning); wz lists every block.
template <typename T, class BatchLoader>
static void xfirst_passes(Context& ctx, c2<T>* base, const BatchLoader& load,
                          const double* kcut2, const int2* wx, int nx, const int2* wy,
                          int ny, const int2* wz, int nz, double bx, double by, double bz) {
  const Geom& g = ctx.g;
  if (nx > 0) {
    if (fast_axis(g.n[0])) {
      TRVG_LOGN_SWITCH(ilog2(g.n[0]), (launch_x_load_batch<T, LG>(
          ctx, base, load, prune_zy(g), kcut2, wx, nx, bx)));
    } else {
      launch_x_load_batch_gen<T>(ctx, base, load, prune_zy(g), kcut2, wx, nx, bx);
    }
  }
  xfirst_yz<T>(ctx, base, kcut2, wy, ny, wz, nz, by, bz);
}

// The y and z passes of a batched x-first transform.
template <typename T>
static void xfirst_yz(Context& ctx, c2<T>* base, const double* kcut2, const int2* wy, int ny,
                      const int2* wz, int nz, double by, double bz) {
  const Geom& g = ctx.g;
  const Prune pr = prune_zy(g);
  if (ny > 0) {
    if (fast_axis(g.n[1])) {
      TRVG_LOGN_SWITCH(ilog2(g.n[1]), (launch_strided_batch<T, LG>(
          ctx, base, g.n[2], (long long)g.n[1] * g.n[2], g.n[2], +1, pr, kcut2, wy, ny, 3,
          by)));
    } else {
      launch_strided_batch_gen<T>(ctx, base, g.n[1], g.n[2], (long long)g.n[1] * g.n[2],
                                  g.n[2], +1, pr, kcut2, wy, ny, 3, by);
    }
  }
  // z pass over every block, reading only the k_z rows the y pass wrote.
  Prune off{};
  off.on = 0;
  LoadMaskedZBatch<T> lz{base, g.nmesh, kcut2, g.dk[2], g.n[2]};
  if (nz > 0) {
    if (fast_axis(g.n[2])) {
      TRVG_LOGN_SWITCH(ilog2(g.n[2]), (launch_z_batch<T, LG>(
          ctx, base, lz, +1, off, kcut2, wz, nz, bz)));
    } else {
      launch_z_batch_gen<T>(ctx, base, lz, +1, off, kcut2, wz, nz, bz);
    }
  }
}

// Shell fields of (ell, m) for `bins`: the backward transform of
// y_lm(k^) src(k) / W(k) on each bin's shell, all bins per pass in one
// launch.  Unpacked: field q at base + q * nmesh.  Packed (real shells:
// real source, even l, m = 0): bins q = 2p, 2p + 1 are the real and
// imaginary parts of base + p * nmesh.
// Launch plan of a shell slab transform (bands, pruning radii, work lists
// and profiler byte counts), a function of the geometry and the bins only:
// built once per device and reused by every later call.
struct ShellPlan {
  DevArray<ShellBand> bands;
  DevArray<double> kc;
  DevArray<int2> w;
  int nx = 0, ny = 0, nz = 0;
  double bx = 0., by = 0., bz = 0.;
};

template <typename T>
static std::shared_ptr<const ShellPlan> shell_plan(Context& ctx, const trvg_binning& kb,
                                                   const std::vector<int>& bins,
                                                   const std::vector<int>& nmodes,
                                                   bool packed) {
  const Geom& g = ctx.g;
  const int nf = int(bins.size());
  std::vector<double> key = {double(ctx.dev), double(sizeof(T)), double(packed)};
  for (int a = 0; a < 3; a++) { key.push_back(g.n[a]); key.push_back(g.dk[a]); }
  for (int b : bins) {
    key.push_back(kb.bin_edges[b]);
    key.push_back(kb.bin_edges[b + 1]);
    key.push_back(nmodes[b]);
  }
  static std::mutex mu;
  static std::map<std::vector<double>, std::shared_ptr<const ShellPlan>> cache;
  {
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
  }
  const int nt = packed ? (nf + 1) / 2 : nf;
  const int per = packed ? 2 : 1;
  const int nl_x = lines_strided<T>(g.n[0]), nl_y = lines_strided<T>(g.n[1]);
  const ShellBand none{HUGE_VAL, HUGE_VAL};
  std::vector<ShellBand> bands((size_t)nt * per, none);
  std::vector<double> kc(nt, 0.);
  // z blocks: every (i, j) line of the last pass.
  const long long nblk = blocks_of((long long)g.n[0] * g.n[1], lines_z(g.n[2]));
  std::vector<int2> wx, wy, wz;
  const double cb = sizeof(c2<T>);
  auto pl = std::make_shared<ShellPlan>();
  for (int q = 0; q < nf; q++) {
    const int b = bins[q];
    bands[q] = shell_band(kb.bin_edges[b], kb.bin_edges[b + 1]);
    Prune pq = make_prune(g, kb.bin_edges[b + 1]);
    kc[q / per] = std::max(kc[q / per], pq.on ? pq.kcut2 : HUGE_VAL);
    pl->bx += double(nmodes[b]) * sizeof(double2);
  }
  for (int f = 0; f < nt; f++) {
    const PruneListsXF& px = prune_lists_xfirst(g, kc[f], nl_x, nl_y);
    for (int w : px.xblocks) wx.push_back(make_int2(f, w));
    for (int w : px.yblocks) wy.push_back(make_int2(f, w));
    for (long long w = 0; w < nblk; w++) wz.push_back(make_int2(f, int(w)));
    const double xw = px.x_lines * g.n[0] * cb;
    const double yw = px.y_lines * g.n[1] * cb;
    pl->bx += xw;
    pl->by += xw + yw;
    pl->bz += yw + double(g.nmesh) * cb;
  }
  pl->nx = int(wx.size());
  pl->ny = int(wy.size());
  pl->nz = int(wz.size());
  pl->bands.reset(bands.size());
  pl->kc.reset(nt);
  pl->w.reset(wx.size() + wy.size() + wz.size());
  wx.insert(wx.end(), wy.begin(), wy.end());
  wx.insert(wx.end(), wz.begin(), wz.end());
  TRVG_HIP(hipMemcpyAsync(pl->bands.get(), bands.data(), bands.size() * sizeof(ShellBand),
                          hipMemcpyHostToDevice, ctx.stream));
  TRVG_HIP(hipMemcpyAsync(pl->kc.get(), kc.data(), nt * sizeof(double),
                          hipMemcpyHostToDevice, ctx.stream));
  TRVG_HIP(hipMemcpyAsync(pl->w.get(), wx.data(), wx.size() * sizeof(int2),
                          hipMemcpyHostToDevice, ctx.stream));
  TRVG_HIP(hipStreamSynchronize(ctx.stream));
  std::lock_guard<std::mutex> lk(mu);
  if (cache.size() >= 64) cache.clear();   // bounded; plans in use stay alive
  cache[key] = pl;
  return pl;
}

template <typename T, typename S>
void shell_slab_ifft(Context& ctx, c2<T>* base, const c2<S>* src,
                     const trvg_binning& kb, const std::vector<int>& bins,
                     const std::vector<int>& nmodes, int ell, int m, bool packed) {
  const Geom& g = ctx.g;
  if (bins.empty()) return;
  const std::shared_ptr<const ShellPlan> pl = shell_plan<T>(ctx, kb, bins, nmodes, packed);
  // The plan outlives the queued launches even if the cache drops it.
  ctx.keep.push_back(std::const_pointer_cast<ShellPlan>(pl));
  const int2* px = pl->w.get();
  const int2* py = px + pl->nx;
  const int2* pz = py + pl->ny;
  if (packed) {
    LoadShellPairBatch<T, S> ld{src, ctx.tab, g, pl->bands.get(), ell, m};
    xfirst_passes<T>(ctx, base, ld, pl->kc.get(), px, pl->nx, py, pl->ny, pz, pl->nz,
                     pl->bx, pl->by, pl->bz);
  } else {
    LoadShellBatch<T, S> ld{src, ctx.tab, g, pl->bands.get(), ell, m};
    xfirst_passes<T>(ctx, base, ld, pl->kc.get(), px, pl->nx, py, pl->ny, pz, pl->nz,
                     pl->bx, pl->by, pl->bz);
  }
}

// Forward transforms in place of the nf meshes at `base`, all of them per
// pass in one launch (work lists cached per device, geometry and nf).
template <typename T>
void slab_fft(Context& ctx, c2<T>* base, int nf) {
  const Geom& g = ctx.g;
  std::vector<double> key = {double(ctx.dev), double(sizeof(T)), double(nf)};
  for (int a = 0; a < 3; a++) key.push_back(g.n[a]);
  static std::mutex mu;
  static std::map<std::vector<double>, std::shared_ptr<ShellPlan>> cache;
  std::shared_ptr<ShellPlan> plan;
  {
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find(key);
    if (it != cache.end()) plan = it->second;
  }
  if (!plan) {
    std::vector<int2> w, wy, wz;
    full_work<T>(g, nf, wz, wy, w);
    plan = std::make_shared<ShellPlan>();
    plan->nx = int(w.size());
    plan->ny = int(wy.size());
    plan->nz = int(wz.size());
    w.insert(w.end(), wy.begin(), wy.end());
    w.insert(w.end(), wz.begin(), wz.end());
    const std::vector<double> kc(nf, HUGE_VAL);
    plan->kc.reset(nf);
    plan->w.reset(w.size());
    TRVG_HIP(hipMemcpyAsync(plan->kc.get(), kc.data(), nf * sizeof(double),
                            hipMemcpyHostToDevice, ctx.stream));
    TRVG_HIP(hipMemcpyAsync(plan->w.get(), w.data(), w.size() * sizeof(int2),
                            hipMemcpyHostToDevice, ctx.stream));
    TRVG_HIP(hipStreamSynchronize(ctx.stream));
    std::lock_guard<std::mutex> lk(mu);
    if (cache.size() >= 16) cache.clear();   // bounded; plans in use stay alive
    cache[key] = plan;
  }
  ctx.keep.push_back(plan);
  const int2* wx = plan->w.get();
  const int2* wy = wx + plan->nx;
  const int2* wz = wy + plan->ny;
  fft3d_batch<T>(ctx, base, LoadSameBatch<T>{base, g.nmesh}, -1, false, plan->kc.get(), wz,
                 plan->nz, wy, plan->ny, wx, plan->nx);
}

template <typename T, int LOGN>
static void launch_x_sjl(Context& ctx, c2<T>* base, int nt, const double2* src,
                         const Spline& sp, const double* r, int ell, int m, bool packed,
                         bool far, double bytes) {
  const Geom& g = ctx.g;
  const unsigned grid =
      unsigned(blocks_of((long long)g.n[1] * g.n[2], strided_lines<T, LOGN>()));
  ProfScope ps(ctx, sizeof(T) == 8 ? KC_FFT_STRIDED64 : KC_FFT_STRIDED, bytes);
  auto kern = packed ? (far ? fft_x_sjl_multi<T, LOGN, true, true>
                            : fft_x_sjl_multi<T, LOGN, true, false>)
                     : (far ? fft_x_sjl_multi<T, LOGN, false, true>
                            : fft_x_sjl_multi<T, LOGN, false, false>);
  raise_lds(kern, strided_smem<T, LOGN>());
  hipLaunchKernelGGL(kern, dim3(grid), dim3(strided_threads<T, LOGN>()),
                     (strided_smem<T, LOGN>()), ctx.stream, base, g.nmesh, nt, src, ctx.tab, g,
                     sp.dev(), r, ell, m, ctx_twiddles<T>(ctx, 1 << LOGN, +1));
  TRVG_LAUNCH_CHECK();
}

template <typename T>
static void launch_x_sjl_gen(Context& ctx, c2<T>* base, int nt, const double2* src,
                             const Spline& sp, const double* r, int ell, int m, bool packed,
                             double bytes) {
  const Geom& g = ctx.g;
  const int N = g.n[0];
  const GenPlan P = make_gen_plan(N);
  const size_t smem = gen_smem<T>(N);
  const unsigned grid = unsigned(blocks_of((long long)g.n[1] * g.n[2], P.nl));
  ProfScope ps(ctx, sizeof(T) == 8 ? KC_FFT_STRIDED64 : KC_FFT_STRIDED, bytes);
  if (packed) {
    auto kern = fft_x_sjl_multi_gen<T, true>;
    raise_lds(kern, smem);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(FFT_THREADS), smem, ctx.stream, base, g.nmesh,
                       nt, src, ctx.tab, g, sp.dev(), r, ell, m,
                       gen_twiddles<T>(ctx, P, +1), P);
  } else {
    auto kern = fft_x_sjl_multi_gen<T, false>;
    raise_lds(kern, smem);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(FFT_THREADS), smem, ctx.stream, base, g.nmesh,
                       nt, src, ctx.tab, g, sp.dev(), r, ell, m,
                       gen_twiddles<T>(ctx, P, +1), P);
  }
  TRVG_LAUNCH_CHECK();
}

// j_l-weighted shell fields of (ell, m) for `bins` (3PCF,
// inv_fourier_transform_sjl_ylm_wgtd_field, field.cpp:1908-2010), r the
// bins' effective radii: x-first batched transforms over every block (no
// band limit); layout and packing as shell_slab_ifft.
template <typename T>
void sjl_slab_ifft(Context& ctx, c2<T>* base, const double2* src, const Spline& sp,
                   const std::vector<double>& r, const std::vector<int>& bins, int ell,
                   int m, bool packed) {
  const Geom& g = ctx.g;
  const int nf = int(bins.size());
  if (nf == 0) return;
  const int nt = packed ? (nf + 1) / 2 : nf;
  const int per = packed ? 2 : 1;
  std::vector<double> rr((size_t)nt * per, -1.);
  for (int q = 0; q < nf; q++) rr[q] = r[bins[q]];
  DevArray<double> dr(rr.size());
  ctx.upload(dr.get(), rr.data(), rr.size());
  // Work lists (y blocks, then every z block, per transform) and the
  // unpruned radii depend on the geometry and the transform count only:
  // built once per device.
  std::vector<double> key = {double(ctx.dev), double(sizeof(T)), double(nt)};
  for (int a = 0; a < 3; a++) key.push_back(g.n[a]);
  static std::mutex mu;
  static std::map<std::vector<double>, std::shared_ptr<ShellPlan>> cache;
  std::shared_ptr<ShellPlan> plan;
  {
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find(key);
    if (it != cache.end()) plan = it->second;
  }
  if (!plan) {
    const PruneListsXF& pl = prune_lists_xfirst(g, HUGE_VAL, lines_strided<T>(g.n[0]),
                                                lines_strided<T>(g.n[1]));
    const long long nblk = blocks_of((long long)g.n[0] * g.n[1], lines_z(g.n[2]));
    std::vector<double> kc(nt, HUGE_VAL);
    std::vector<int2> w;   // y blocks, then z blocks
    for (int f = 0; f < nt; f++)
      for (int b : pl.yblocks) w.push_back(make_int2(f, b));
    const size_t ny = w.size();
    for (int f = 0; f < nt; f++)
      for (long long b = 0; b < nblk; b++) w.push_back(make_int2(f, int(b)));
    plan = std::make_shared<ShellPlan>();
    plan->ny = int(ny);
    plan->nz = int(w.size() - ny);
    plan->kc.reset(nt);
    plan->w.reset(w.size());
    TRVG_HIP(hipMemcpyAsync(plan->kc.get(), kc.data(), nt * sizeof(double),
                            hipMemcpyHostToDevice, ctx.stream));
    TRVG_HIP(hipMemcpyAsync(plan->w.get(), w.data(), w.size() * sizeof(int2),
                            hipMemcpyHostToDevice, ctx.stream));
    TRVG_HIP(hipStreamSynchronize(ctx.stream));
    std::lock_guard<std::mutex> lk(mu);
    if (cache.size() >= 16) cache.clear();   // bounded; plans in use stay alive
    cache[key] = plan;
  }
  ctx.keep.push_back(plan);
  const size_t ny = size_t(plan->ny), nz = size_t(plan->nz);
  const int2* dwp = plan->w.get();
  // Algorithmic bytes: the source read once, then each pass writes (and the
  // later ones read) every field.
  const double fb = double(g.nmesh) * sizeof(c2<T>) * nt;
  const double bx = double(g.nmesh) * sizeof(double2) + fb, by = 2. * fb, bz = 2. * fb;
  // Whether some argument |k| r leaves the spline's range.
  double k2 = 0., rmax = 0.;
  for (int a = 0; a < 3; a++) k2 += std::pow(g.n[a] / 2 * g.dk[a], 2);
  for (double v : rr) rmax = std::max(rmax, v);
  const bool far = !(std::sqrt(k2) * rmax * (1. + 1.e-9) < sp.split);
  if (fast_axis(g.n[0])) {
    TRVG_LOGN_SWITCH(ilog2(g.n[0]), (launch_x_sjl<T, LG>(ctx, base, nt, src, sp, dr.get(),
                                                          ell, m, packed, far, bx)));
  } else {
    launch_x_sjl_gen<T>(ctx, base, nt, src, sp, dr.get(), ell, m, packed, bx);
  }
  // The radii stay owned until the stream is synchronised: returned to the
  // shared pool now, another call could take and overwrite them while the
  // x pass still reads them.
  ctx.keep_until_flush(std::move(dr));
  xfirst_yz<T>(ctx, base, plan->kc.get(), dwp, int(ny), dwp + ny, int(nz), by, bz);
}

template <typename T, class Loader>
void fft3d(Context& ctx, c2<T>* data, const Loader& load, int sign,
           double read_bytes, const Prune* prune) {
  const Geom& g = ctx.g;
  Prune pr{};
  pr.on = 0;
  if (prune) pr = *prune;
  const double cb = sizeof(c2<T>);
  // Lines / slabs each pass touches (for the profiler's algorithmic bytes).
  double d_lines = double(g.n[0]) * g.n[1], slabs = g.n[0];
  if (pr.on) {
    d_lines = 0.;
    slabs = 0.;
    for (int i = 0; i < g.n[0]; i++) {
      double kx = shifted(i, g.n[0]) * g.dk[0];
      if (kx * kx < pr.kcut2) slabs += 1.;
      for (int j = 0; j < g.n[1]; j++) {
        double ky = shifted(j, g.n[1]) * g.dk[1];
        if (kx * kx + ky * ky < pr.kcut2) d_lines += 1.;
      }
    }
  }
  if (read_bytes < 0.) read_bytes = double(g.nmesh) * cb;
  const double zw = d_lines * g.n[2] * cb;
  const double slab_vals = slabs * g.n[1] * g.n[2];
  if (fast_axis(g.n[2])) {
    TRVG_LOGN_SWITCH(ilog2(g.n[2]), (launch_z<T, LG, Loader>(
        ctx, data, load, sign, read_bytes, zw, pr)));
  } else {
    launch_z_gen<T>(ctx, data, load, sign, read_bytes + zw, pr);
  }
  if (fast_axis(g.n[1])) {
    TRVG_LOGN_SWITCH(ilog2(g.n[1]), (launch_strided<T, LG>(
        ctx, data, g.n[2], (long long)g.n[1] * g.n[2], g.n[2], sign, pr, 1,
        zw + slab_vals * cb)));
  } else {
    launch_strided_gen<T>(ctx, data, g.n[1], g.n[2], (long long)g.n[1] * g.n[2], g.n[2],
                          sign, pr, 1, zw + slab_vals * cb);
  }
  if (fast_axis(g.n[0])) {
    TRVG_LOGN_SWITCH(ilog2(g.n[0]), (launch_strided<T, LG>(
        ctx, data, (long long)g.n[1] * g.n[2], 0, (long long)g.n[1] * g.n[2], sign,
        pr, 2, slab_vals * cb + double(g.nmesh) * cb)));
  } else {
    launch_strided_gen<T>(ctx, data, g.n[0], (long long)g.n[1] * g.n[2], 0,
                          (long long)g.n[1] * g.n[2], sign, pr, 2,
                          slab_vals * cb + double(g.nmesh) * cb);
  }
}

}  // namespace trvg

// engine_drivers.hip -- estimator drivers of the gfx950 engine.
//
// The drivers compute what src/triumvirate/src/threept.cpp computes, term by
// term in the same (m1, m2, M) enumeration, but each distinct quantity once:
//   * one shell-filtered IFFT per distinct (bin, side) instead of two per
//     bin pair (threept.cpp:664-669, 725-730);
//   * one shot-noise IFFT per term instead of one per bin pair
//     (field.cpp:3269-3345 called at threept.cpp:950-964), followed by a
//     radial histogram so each pair costs O(#radii) spline evaluations;
//   * G_LM and the shot-noise field dn_LM share one assignment + FFT
//     (threept.cpp:452-457, 777-784), and for (L, M) = (0, 0) both are the
//     already-transformed dn_00.
// Results differ from the reference only by floating-point summation order.
#include <algorithm>
#include <cstring>
#include <map>
#include <set>
#include <tuple>
#include <type_traits>

#include "engine.hpp"

namespace trvg {

// ---------------------------------------------------------------------------
// Small launch helpers
// ---------------------------------------------------------------------------

template <typename T>
static void zero_field(Context& ctx, c2<T>* f) {
  ProfScope ps(ctx, KC_MISC, double(ctx.g.nmesh) * sizeof(c2<T>));
  hipLaunchKernelGGL((k_zero<T>), dim3(grid_for(ctx, ctx.g.nmesh)),
                     dim3(RED_THREADS), 0, ctx.stream, f, ctx.g.nmesh);
  TRVG_LAUNCH_CHECK();
}

TileSorter::TileSorter(Context& ctx, const DeviceCatalogue& c)
    : ctx_(ctx), c_(c), tv_(std::make_unique<TiledView>()) {
  const Geom& g = ctx.g;
  for (int a = 0; a < 3; a++) {
    tv_->n[a] = g.n[a];
    tv_->L[a] = g.L[a];
    tv_->tg.nt[a] = (g.n[a] + TILE - 1) / TILE;
  }
  tv_->tg.ntiles = (long long)tv_->tg.nt[0] * tv_->tg.nt[1] * tv_->tg.nt[2];
  const long long nt = tv_->tg.ntiles;
  tile_of_.reset(c.n);
  key2_.reset(c.n);
  ccount_.reset((nt + 1) * TILE_CLASSES);
  TRVG_HIP(hipMemsetAsync(ccount_.get(), 0, (nt + 1) * TILE_CLASSES * 4, ctx.stream));
}

void TileSorter::count(long long begin, long long end) {
  if (end <= begin) return;
  ProfScope ps(ctx_, KC_ASSIGN, double(end - begin) * 32.);
  hipLaunchKernelGGL(k_tile_count, dim3(grid_for(ctx_, end - begin, 16)), dim3(256), 0,
                     ctx_.stream, c_.view(), begin, end, ctx_.g, tv_->tg, tile_of_.get(),
                     ccount_.get(), key2_.get());
  TRVG_LAUNCH_CHECK();
}

void TileSorter::finish(bool move_w, bool move_los) {
  Context& ctx = ctx_;
  const DeviceCatalogue& c = c_;
  move_los = move_los && c.los.get() != nullptr;
  const long long nt = tv_->tg.ntiles;
  DevArray<unsigned int> counts(nt + 1), offs(nt + 2), nch(nt), woff(nt + 1);
  hipLaunchKernelGGL(k_tile_sum, dim3(grid_for(ctx, nt + 1)), dim3(256), 0, ctx.stream,
                     ccount_.get(), nt + 1, counts.get());
  hipLaunchKernelGGL(k_scan_counts, dim3(1), dim3(1024), 0, ctx.stream,
                     counts.get(), nt + 1, offs.get());
  TRVG_LAUNCH_CHECK();
  DevArray<double> sx(c.n), sy(c.n), sz(c.n), sw(move_w ? c.n : 0),
      slos(move_los ? 3 * c.n : 0);
  {
    ProfScope ps(ctx, KC_ASSIGN, c.n * (20. + 48. + (move_w ? 16. : 0.) + (move_los ? 48. : 0.)));
    DevArray<double2> rec(2 * size_t(c.n));
    hipLaunchKernelGGL(k_tile_scatter, dim3(grid_for(ctx, c.n, 16)), dim3(256), 0,
                       ctx.stream, c.view(), tile_of_.get(), offs.get(), ccount_.get(),
                       key2_.get(), rec.get(), move_w, slos.get());
    hipLaunchKernelGGL(k_tile_columns, dim3(grid_for(ctx, c.n, 16)), dim3(256), 0,
                       ctx.stream, rec.get(), c.n, sx.get(), sy.get(), sz.get(), sw.get());
    TRVG_LAUNCH_CHECK();
    ctx.keep_until_flush(std::move(rec));
  }
  // Work list: chunks of at most TILE_CHUNK particles per tile.
  tv_->work_cap = nt + (c.n + TILE_CHUNK - 1) / TILE_CHUNK;
  tv_->work.reset(tv_->work_cap);
  tv_->meta.reset(2);
  const unsigned tgrid = grid_for(ctx, nt);
  hipLaunchKernelGGL(k_tile_chunks, dim3(tgrid), dim3(256), 0, ctx.stream, offs.get(),
                     nt, nch.get());
  hipLaunchKernelGGL(k_scan_counts, dim3(1), dim3(1024), 0, ctx.stream, nch.get(), nt,
                     woff.get());
  hipLaunchKernelGGL(k_tile_work, dim3(tgrid), dim3(256), 0, ctx.stream, offs.get(),
                     woff.get(), nt, tv_->work.get(), tv_->meta.get());
  TRVG_LAUNCH_CHECK();
  // The permuted columns replace the caller-order ones; the old columns and
  // the sort's temporaries stay allocated until the stream has passed them.
  std::swap(c.x, sx); std::swap(c.y, sy); std::swap(c.z, sz);
  if (move_w) std::swap(c.w, sw);
  if (move_los) std::swap(c.los, slos);
  ctx.keep_until_flush(std::move(sx)); ctx.keep_until_flush(std::move(sy));
  ctx.keep_until_flush(std::move(sz)); ctx.keep_until_flush(std::move(sw));
  ctx.keep_until_flush(std::move(slos));
  ctx.keep_until_flush(std::move(tile_of_)); ctx.keep_until_flush(std::move(counts));
  ctx.keep_until_flush(std::move(offs)); ctx.keep_until_flush(std::move(ccount_));
  ctx.keep_until_flush(std::move(key2_)); ctx.keep_until_flush(std::move(nch));
  ctx.keep_until_flush(std::move(woff));
  // Exact grids for later calls once the host has the counts.
  const unsigned int* hm = ctx.download(tv_->meta.get(), 2);
  TiledView* tvp = tv_.get();
  const long long n = c.n;
  ctx.defer([tvp, hm, n] {
    tvp->nwork = hm[0];
    tvp->nstraggle = n - (long long)hm[1];
  });
  c.tiled = std::move(tv_);
}

// Tile order of `c` for the context's mesh (built once per geometry and
// cached on the catalogue): a counting sort by tile with the within-tile
// bank-class order, the columns permuted in place, and the work list built
// on the device.  Nothing here waits for the device.
static const TiledView& tiled_view(Context& ctx, const DeviceCatalogue& c) {
  if (c.tiled && c.tiled->matches(ctx.g)) return *c.tiled;
  TileSorter ts(ctx, c);
  ts.count(0, c.n);
  ts.finish();
  return *c.tiled;
}

// Grid of the tiled kernels: the exact work count once known, else the bound.
static unsigned tile_grid(const TiledView& tv) {
  return unsigned(tv.nwork >= 0 ? tv.nwork : tv.work_cap);
}

template <typename T, int ORDER>
static void assign_order(Context& ctx, c2<T>* mesh, const DeviceCatalogue& c,
                         const TiledView& tv, int mode, int ell, int m, double scale,
                         int cplx_w, bool shadow) {
  DevParticles sv = c.view();
  if (tile_grid(tv) > 0) {
    auto kern = cplx_w == 1 ? (shadow ? k_assign_tiled<T, ORDER, true, true>
                                      : k_assign_tiled<T, ORDER, true, false>)
                            : (shadow ? k_assign_tiled<T, ORDER, false, true>
                                      : k_assign_tiled<T, ORDER, false, false>);
    hipLaunchKernelGGL(kern, dim3(tile_grid(tv)), dim3(256), 0, ctx.stream, mesh, sv, ctx.g,
                       tv.tg, tv.work.get(), tv.meta.get(), mode, ell, m, scale, cplx_w);
    TRVG_LAUNCH_CHECK();
  }
  // Stragglers [meta[1], n) keep the reference's flattened-index rule.
  if (tv.nstraggle != 0) {
    hipLaunchKernelGGL((k_assign<T, ORDER>), dim3(tv.nstraggle > 0
                                                      ? grid_for(ctx, tv.nstraggle, 16)
                                                      : 64u),
                       dim3(256), 0, ctx.stream, mesh, sv, ctx.g, mode, ell, m, scale,
                       cplx_w, int(shadow), tv.meta.get() + 1);
    TRVG_LAUNCH_CHECK();
  }
}

// imag: a real weight (m = 0 or a unit/scalar mode) goes into the
// imaginary parts of the mesh instead of the real parts.  shadow: the
// half-cell-shifted pass of interlacing.
template <typename T>
static void assign(Context& ctx, c2<T>* mesh, const DeviceCatalogue& c,
                   int mode, int ell, int m, double scale, bool imag = false,
                   bool shadow = false) {
  // y_l0 is real (its imaginary part is a signed zero): m = 0 fields take
  // real parts only.
  int cplx_w = ((mode == WM_YLM_W || mode == WM_YLMC_W2) && m != 0);
  if (imag) {
    if (cplx_w) throw Error(TRVG_ERR_INTERNAL, "Complex weights have no imaginary slot.");
    cplx_w = 2;
  }
  if ((mode == WM_YLM_W || mode == WM_YLMC_W2) && c.los.get() == nullptr)
    throw Error(TRVG_ERR_DATA, "Lines of sight are required for survey-type fields.");
  const TiledView& tv = tiled_view(ctx, c);
  // Algorithmic bytes: particle columns read once (position, weight,
  // line of sight when used) plus one write of the mesh.
  double pbytes = 24. + (mode == WM_UNIT ? 0. : 8.) +
                  ((mode == WM_YLM_W || mode == WM_YLMC_W2) ? 24. : 0.);
  ProfScope ps(ctx, KC_ASSIGN, c.n * pbytes + double(ctx.g.nmesh) * sizeof(c2<T>));
  switch (ctx.p.assignment_order) {
    case 1: assign_order<T, 1>(ctx, mesh, c, tv, mode, ell, m, scale, cplx_w, shadow); break;
    case 2: assign_order<T, 2>(ctx, mesh, c, tv, mode, ell, m, scale, cplx_w, shadow); break;
    case 3: assign_order<T, 3>(ctx, mesh, c, tv, mode, ell, m, scale, cplx_w, shadow); break;
    default: assign_order<T, 4>(ctx, mesh, c, tv, mode, ell, m, scale, cplx_w, shadow); break;
  }
}

template <typename T, int ORDER>
static void assign_dual_order(Context& ctx, T* ra, T* rb, const DeviceCatalogue& c,
                              const TiledView& tv, int ell, int m, double scale_a,
                              double scale_b) {
  DevParticles sv = c.view();
  const bool cplx = m != 0;
  if (tile_grid(tv) > 0) {
    const size_t smem = size_t(cplx ? 4 : 2) * TILE_CELLS * sizeof(double);
    if (cplx)
      hipLaunchKernelGGL((k_assign_tiled_dual<T, ORDER, true>), dim3(tile_grid(tv)),
                         dim3(256), smem, ctx.stream, ra, rb, sv, ctx.g, tv.tg,
                         tv.work.get(), tv.meta.get(), ell, m, scale_a, scale_b);
    else
      hipLaunchKernelGGL((k_assign_tiled_dual<T, ORDER, false>), dim3(tile_grid(tv)),
                         dim3(256), smem, ctx.stream, ra, rb, sv, ctx.g, tv.tg,
                         tv.work.get(), tv.meta.get(), ell, m, scale_a, scale_b);
    TRVG_LAUNCH_CHECK();
  }
  if (tv.nstraggle != 0) {
    // Real outputs sharing one mesh (rb = ra + 1): B goes to imaginary parts.
    const bool shared = rb == ra + 1;
    c2<T>* ma = reinterpret_cast<c2<T>*>(ra);
    c2<T>* mb = shared ? ma : reinterpret_cast<c2<T>*>(rb);
    const int cwa = cplx ? 1 : 0, cwb = cplx ? 1 : (shared ? 2 : 0);
    const unsigned sg = tv.nstraggle > 0 ? grid_for(ctx, tv.nstraggle, 16) : 64u;
    hipLaunchKernelGGL((k_assign<T, ORDER>), dim3(sg), dim3(256), 0, ctx.stream, ma, sv,
                       ctx.g, WM_YLM_W, ell, m, scale_a, cwa, 0, tv.meta.get() + 1);
    hipLaunchKernelGGL((k_assign<T, ORDER>), dim3(sg), dim3(256), 0, ctx.stream, mb, sv,
                       ctx.g, WM_YLMC_W2, ell, m, scale_b, cwb, 0, tv.meta.get() + 1);
    TRVG_LAUNCH_CHECK();
  }
}

// A += scale_a sum y_lm w W / V_cell and B += scale_b sum y_lm^* w^2 W /
// V_cell over catalogue c in one pass (survey catalogues: lines of sight
// needed); ra, rb point at the real part of cell 0 of each output.
template <typename T>
static void assign_dual(Context& ctx, T* ra, T* rb, const DeviceCatalogue& c, int ell,
                        int m, double scale_a, double scale_b) {
  if (c.los.get() == nullptr)
    throw Error(TRVG_ERR_DATA, "Lines of sight are required for survey-type fields.");
  const TiledView& tv = tiled_view(ctx, c);
  // Algorithmic bytes: position, weight and line of sight read once, the
  // output values written once.
  const double outb = (m != 0 ? 2. : 1.) * double(ctx.g.nmesh) * sizeof(c2<T>);
  ProfScope ps(ctx, KC_ASSIGN, c.n * 56. + outb);
  switch (ctx.p.assignment_order) {
    case 1: assign_dual_order<T, 1>(ctx, ra, rb, c, tv, ell, m, scale_a, scale_b); break;
    case 2: assign_dual_order<T, 2>(ctx, ra, rb, c, tv, ell, m, scale_a, scale_b); break;
    case 3: assign_dual_order<T, 3>(ctx, ra, rb, c, tv, ell, m, scale_a, scale_b); break;
    default: assign_dual_order<T, 4>(ctx, ra, rb, c, tv, ell, m, scale_a, scale_b); break;
  }
}

template <typename T>
void assign_add(Context& ctx, c2<T>* mesh, const DeviceCatalogue& c, int mode,
                int ell, int m, double scale, bool shadow) {
  assign<T>(ctx, mesh, c, mode, ell, m, scale, false, shadow);
}
template void assign_add<double>(Context&, double2*, const DeviceCatalogue&, int, int,
                                 int, double, bool);

template <typename T>
void assign_field(Context& ctx, c2<T>* mesh, const DeviceCatalogue& c, int mode,
                  int ell, int m, double scale) {
  zero_field<T>(ctx, mesh);
  assign<T>(ctx, mesh, c, mode, ell, m, scale);
}
template void assign_field<double>(Context&, double2*, const DeviceCatalogue&,
                                   int, int, int, double);
template void assign_field<float>(Context&, float2*, const DeviceCatalogue&,
                                  int, int, int, double);

// Survey field  sum_d y w - alpha sum_r y w  (quad: conj(y) w^2 with
// +alpha^2), or box field (unit weights, optional mean subtraction), then
// the forward transform with the V_cell factor.
template <typename T>
static void build_field_k(Context& ctx, c2<T>* f, const DeviceCatalogue& d,
                          const DeviceCatalogue* r, bool survey, double alpha,
                          int ell, int m, bool quad, bool fluctuation) {
  zero_field<T>(ctx, f);
  T shift = T(0);
  if (survey) {
    int mode = quad ? WM_YLMC_W2 : WM_YLM_W;
    assign<T>(ctx, f, d, mode, ell, m, 1.);
    assign<T>(ctx, f, *r, mode, ell, m, quad ? alpha * alpha : -alpha);
  } else {
    assign<T>(ctx, f, d, WM_UNIT, 0, 0, 1.);
    if (fluctuation) shift = T(-(double(d.n) / ctx.g.vol));
  }
  LoadScaleShift<T> ld{f, shift, T(ctx.g.vol_cell)};
  fft3d<T>(ctx, f, ld, -1);
}

// One catalogue's field alpha sum_c y w (quad: alpha^2 sum_c y^* w^2),
// forward transformed with the V_cell factor (field.cpp:1325-1362,
// 1449-1489).
static void build_single_field_k(Context& ctx, double2* f, const DeviceCatalogue& c,
                                 double alpha, int ell, int m, bool quad) {
  zero_field<double>(ctx, f);
  assign<double>(ctx, f, c, quad ? WM_YLMC_W2 : WM_YLM_W, ell, m,
                 quad ? alpha * alpha : alpha);
  LoadScaleShift<double> ld{f, 0., ctx.g.vol_cell};
  fft3d<double>(ctx, f, ld, -1);
}

// Survey pair of one (l, m): the density contrast
//   dn = sum_d y w - alpha sum_r y w
// and its shot-noise field
//   N = sum_d y^* w^2 + alpha^2 sum_r y^* w^2,
// both assigned in one pass per catalogue and forward transformed.  For
// m = 0 both fields are real: they are assigned as dn + i N into one mesh,
// transformed once and separated by Hermitian symmetry.  `data_assigned`
// (catalogues of uniform weights only): dn already holds S_d, as
// prefill_survey_data leaves it.
static void build_survey_pair_k(Context& ctx, double2* dn, double2* N,
                                const DeviceCatalogue& d, const DeviceCatalogue& r,
                                double alpha, int ell, int m,
                                bool data_assigned = false) {
  double* rdn = reinterpret_cast<double*>(dn);
  // Catalogues of uniform weights: one accumulation per particle, S_c =
  // sum_c y w W, and the pair from the transforms by linearity (for a
  // uniform w, y^* w^2 = w (y w)^*).
  const bool uniform = std::isfinite(d.wuni) && std::isfinite(r.wuni);
  if (data_assigned && !uniform)
    throw Error(TRVG_ERR_PARAM, "Prefilled data fields need uniform weights.");
  if (m == 0) {
    if (uniform) {
      if (!data_assigned) {
        zero_field<double>(ctx, dn);
        assign<double>(ctx, dn, d, WM_YLM_W, ell, 0, 1.);
      }
      assign<double>(ctx, dn, r, WM_YLM_W, ell, 0, 1., true);
    } else {
      zero_field<double>(ctx, dn);
      assign_dual<double>(ctx, rdn, rdn + 1, d, ell, m, 1., 1.);
      assign_dual<double>(ctx, rdn, rdn + 1, r, ell, m, -alpha, alpha * alpha);
    }
    LoadScaleShift<double> la{dn, 0., ctx.g.vol_cell};
    fft3d<double>(ctx, dn, la, -1);
    ProfScope ps(ctx, KC_MISC, 3. * double(ctx.g.nmesh) * sizeof(double2));
    // Plain separation (dn + i N), or dn = S_d - alpha S_r and
    // N = w_d S_d + alpha^2 w_r S_r from S_d + i S_r.
    const double pa = 1., pb = uniform ? -alpha : 0.;
    const double qa = uniform ? d.wuni : 0., qb = uniform ? alpha * alpha * r.wuni : 1.;
    hipLaunchKernelGGL(k_unpack_hermitian, dim3(grid_for(ctx, ctx.g.nmesh)), dim3(256), 0,
                       ctx.stream, dn, N, ctx.g, pa, pb, qa, qb);
    TRVG_LAUNCH_CHECK();
    return;
  }
  if (uniform) {
    // S_d in dn, S_r in a scratch mesh; N (out of place) first, then dn in
    // place over S_d, each formed by its transform's first-pass loader.
    DevArray<double2> sr(ctx.g.nmesh);
    if (!data_assigned) zero_field<double>(ctx, dn);
    zero_field<double>(ctx, sr.get());
    if (!data_assigned) assign<double>(ctx, dn, d, WM_YLM_W, ell, m, 1.);
    assign<double>(ctx, sr.get(), r, WM_YLM_W, ell, m, 1.);
    const double vc = ctx.g.vol_cell, rb2 = 2. * double(ctx.g.nmesh) * sizeof(double2);
    LoadLinear2<double> lb{dn, sr.get(), d.wuni * vc, alpha * alpha * r.wuni * vc, 1};
    fft3d<double>(ctx, N, lb, -1, rb2);
    LoadLinear2<double> la{dn, sr.get(), vc, -alpha * vc, 0};
    fft3d<double>(ctx, dn, la, -1, rb2);
    ctx.keep_until_flush(std::move(sr));
    return;
  }
  zero_field<double>(ctx, dn);
  zero_field<double>(ctx, N);
  assign_dual<double>(ctx, rdn, reinterpret_cast<double*>(N), d, ell, m, 1., 1.);
  assign_dual<double>(ctx, rdn, reinterpret_cast<double*>(N), r, ell, m, -alpha,
                      alpha * alpha);
  LoadScaleShift<double> la{dn, 0., ctx.g.vol_cell};
  fft3d<double>(ctx, dn, la, -1);
  LoadScaleShift<double> lb{N, 0., ctx.g.vol_cell};
  fft3d<double>(ctx, N, lb, -1);
}

// ---------------------------------------------------------------------------
// Reductions
// ---------------------------------------------------------------------------

// n_modes and k_eff per bin depend on the geometry and the edges only:
// computed once per device and reused.
ShellStats shell_stats(Context& ctx, const trvg_binning& kb) {
  const int nb = kb.num_bins;
  std::vector<double> key = {double(ctx.dev)};
  for (int a = 0; a < 3; a++) { key.push_back(ctx.g.n[a]); key.push_back(ctx.g.dk[a]); }
  key.insert(key.end(), kb.bin_edges, kb.bin_edges + nb + 1);
  static std::mutex mu;
  static std::map<std::vector<double>, ShellStats> cache;
  {
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
  }
  DevArray<double> edges(nb + 1);
  TRVG_HIP(hipMemcpyAsync(edges.get(), kb.bin_edges, (nb + 1) * 8,
                          hipMemcpyHostToDevice, ctx.stream));
  unsigned grid = grid_for(ctx, ctx.g.nmesh, 4);
  DevArray<unsigned long long> cnt(nb);
  DevArray<double> part((size_t)grid * nb), ks(nb);
  TRVG_HIP(hipMemsetAsync(cnt.get(), 0, nb * 8, ctx.stream));
  size_t smem = nb * (8 + 4);
  ProfScope ps(ctx, KC_SHELL_STATS, 0.);
  hipLaunchKernelGGL(k_shell_stats, dim3(grid), dim3(RED_THREADS), smem,
                     ctx.stream, ctx.g, edges.get(), nb, cnt.get(), part.get());
  TRVG_LAUNCH_CHECK();
  reduce_cols(ctx, part.get(), int(grid), nb, ks.get());
  std::vector<unsigned long long> hc(nb);
  ShellStats s;
  s.keff.resize(nb);
  TRVG_HIP(hipMemcpyAsync(hc.data(), cnt.get(), nb * 8, hipMemcpyDeviceToHost, ctx.stream));
  TRVG_HIP(hipMemcpyAsync(s.keff.data(), ks.get(), nb * 8, hipMemcpyDeviceToHost, ctx.stream));
  TRVG_HIP(hipStreamSynchronize(ctx.stream));
  s.nmodes.resize(nb);
  for (int b = 0; b < nb; b++) {
    s.nmodes[b] = int(hc[b]);
    s.keff[b] /= double(s.nmodes[b]);   // NaN for an empty shell, as k_eff /= 0
  }
  std::lock_guard<std::mutex> lk(mu);
  if (cache.size() >= 64) cache.clear();
  cache[key] = s;
  return s;
}

// The two-point binning map: z-line windows and offsets on the host (the
// window only has to contain every cell with |k| <= twopt_kmax), the exact
// bin rule per cell on the device.
std::shared_ptr<const TwoptMapData> twopt_map(Context& ctx, const double* edges, int nb) {
  if (nb < 1 || nb >= int(TWOPT_NONE)) throw std::invalid_argument("twopt_map: bin count");
  std::vector<double> key = {double(ctx.dev)};
  for (int a = 0; a < 3; a++) { key.push_back(ctx.g.n[a]); key.push_back(ctx.g.dk[a]); }
  key.insert(key.end(), edges, edges + nb + 1);
  static std::mutex mu;
  static std::map<std::vector<double>, std::shared_ptr<const TwoptMapData>> cache;
  {
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
  }
  const Geom& g = ctx.g;
  const long long nlines = (long long)g.n[0] * g.n[1];
  const int half = g.n[2] / 2;
  const double kmax = twopt_kmax(edges[nb]);
  std::vector<int> K(nlines);
  std::vector<long long> off(nlines);
  long long tot = 0;
  for (long long l = 0; l < nlines; l++) {
    const double kx = shifted(int(l / g.n[1]), g.n[0]) * g.dk[0];
    const double ky = shifted(int(l % g.n[1]), g.n[1]) * g.dk[1];
    const double rem = kmax * kmax - (kx * kx + ky * ky);
    off[l] = tot;
    if (rem < 0.) { K[l] = -1; continue; }
    K[l] = int(std::sqrt(rem) / g.dk[2]) + 1;
    tot += (K[l] >= half ? half : K[l]) + 1;
  }
  auto d = std::make_shared<TwoptMapData>();
  d->K.reset(nlines);
  d->off.reset(nlines);
  d->bin.reset(tot > 0 ? tot : 1);
  DevArray<double> de(nb + 1);
  TRVG_HIP(hipMemcpyAsync(d->K.get(), K.data(), nlines * sizeof(int), hipMemcpyHostToDevice,
                          ctx.stream));
  TRVG_HIP(hipMemcpyAsync(d->off.get(), off.data(), nlines * sizeof(long long),
                          hipMemcpyHostToDevice, ctx.stream));
  TRVG_HIP(hipMemcpyAsync(de.get(), edges, (nb + 1) * 8, hipMemcpyHostToDevice, ctx.stream));
  hipLaunchKernelGGL(k_twopt_binmap, dim3(grid_for(ctx, nlines * 64, 4)), dim3(RED_THREADS), 0,
                     ctx.stream, g, d->view(), de.get(), nb, d->bin.get());
  TRVG_LAUNCH_CHECK();
  // The host vectors and `de` must outlive the copies and the build.
  TRVG_HIP(hipStreamSynchronize(ctx.stream));
  std::lock_guard<std::mutex> lk(mu);
  if (cache.size() >= 16) cache.clear();   // bounded; maps in use stay alive
  cache[key] = d;
  return d;
}

// Launch of the direct-to-LDS pair kernel (opting in to more than 64 KiB of
// dynamic LDS where a launch needs it).
template <typename T, int MODE>
static void launch_pair_lds(Context& ctx, unsigned grid, size_t smem, const c2<T>* fa,
                            int nas, const c2<T>* fb, int nbs, const c2<T>* G,
                            long long nm, const int2* tiles, int nt, double2* part) {
  if (smem > 64 * 1024)
    TRVG_HIP(hipFuncSetAttribute((const void*)k_pair_lds<T, MODE>,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, int(smem)));
  hipLaunchKernelGGL((k_pair_lds<T, MODE>), dim3(grid), dim3(256), smem, ctx.stream, fa,
                     nas, fb, nbs, G, nm, tiles, nt, part);
  TRVG_LAUNCH_CHECK();
}

// What a term uses of its pair sums S: it adds S + f conj(S), twice the
// real part (f = 1) or the imaginary part (f = -1) of a term counted with its
// mirror, or S itself (f = 0, the term of m1 = m2 = M = 0).
enum PairPart { PAIR_FULL, PAIR_REAL, PAIR_IMAG };
static PairPart wanted(double f_mirror) {
  return f_mirror > 0. ? PAIR_REAL : (f_mirror < 0. ? PAIR_IMAG : PAIR_FULL);
}

template <int MODE, bool FULL, int NTA>
static auto pair_mfma_kernel(int ntb) {
  return ntb == 1 ? k_pair_mfma<MODE, FULL, NTA, 1> : k_pair_mfma<MODE, FULL, NTA, 2>;
}

template <int MODE, bool FULL>
static void launch_pair_mfma(Context& ctx, unsigned grid, size_t smem, const float2* fa,
                             int nas, const float2* fb, int nbs, const float2* G,
                             long long nm, int nta, int ntb, unsigned mask, bool same,
                             bool rot, double* part) {
  auto kern = nta == 1 ? pair_mfma_kernel<MODE, FULL, 1>(ntb) : pair_mfma_kernel<MODE, FULL, 2>(ntb);
  if (smem > 64 * 1024)
    TRVG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, int(smem)));
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256), smem, ctx.stream, fa, nas, fb, nbs, G, nm,
                     mask, int(same), int(rot), part);
  TRVG_LAUNCH_CHECK();
}

// pair_reduce of a table of FP32 fields with a complex A side on the matrix
// cores (k_pair_mfma).
static void pair_reduce_mfma(Context& ctx, const float2* FA, int na, const float2* FB,
                             int nbf, bool b_packed, const float2* G, PairPart want,
                             const std::vector<int2>& pairs,
                             std::function<void(std::vector<cplx>&&)> sink) {
  const int mode = b_packed ? 1 : 0;
  const bool full = want == PAIR_FULL;
  const long long nm = ctx.g.nmesh;
  constexpr int SIDE = PM_TILE * PM_NT;   // fields a side of one launch
  struct Group {
    int a0, b0, nta, ntb;
    const double* h;
  };
  std::vector<Group> groups;
  const long long nchunks = nm / PairLds<float>::LDC;
  for (int b0 = 0; b0 < nbf; b0 += SIDE) {
    for (int a0 = 0; a0 < na; a0 += SIDE) {
      const int nas = std::min(SIDE, na - a0), nbs = std::min(SIDE, nbf - b0);
      const int nta = (nas + PM_TILE - 1) / PM_TILE, ntb = (nbs + PM_TILE - 1) / PM_TILE;
      unsigned mask = 0u;
      for (const int2& pr : pairs)
        if (pr.x >= a0 && pr.x < a0 + nas && pr.y >= b0 && pr.y < b0 + nbs)
          mask |= 1u << ((pr.x - a0) / PM_TILE * ntb + (pr.y - b0) / PM_TILE);
      if (mask == 0u) continue;
      const bool same = FA == FB && !b_packed && a0 == b0 && nas == nbs;
      const int ma = pair_rows_a(mode, nas), mb = same ? 0 : pair_rows_b(mode, nbs);
      const size_t smem = pair_mfma_smem(ma + mb + 1, nta * ntb, full);
      const int per_cu = std::max(1, std::min(8, int((160 * 1024) / smem)));
      const unsigned grid =
          unsigned(std::max<long long>(1, std::min<long long>(nchunks, (long long)ctx.sm_count * per_cu)));
      const int width = nta * ntb * PM_TILE * PM_TILE * (full ? 2 : 1);
      DevArray<double> part((size_t)grid * width), sum(width);
      {
        // A packed side holds two fields per mesh (group starts are even).
        const float2* fa = FA + (long long)a0 * nm;
        const float2* fb = FB + (long long)(mode >= 1 ? b0 / 2 : b0) * nm;
        ProfScope ps(ctx, KC_PAIR_REDUCE, (ma + mb + 1.) * double(nm) * sizeof(float2));
        const bool rot = want == PAIR_IMAG;
        auto go = mode == 1 ? (full ? launch_pair_mfma<1, true> : launch_pair_mfma<1, false>)
                            : (full ? launch_pair_mfma<0, true> : launch_pair_mfma<0, false>);
        go(ctx, grid, smem, fa, nas, fb, nbs, G, nm, nta, ntb, mask, same, rot, part.get());
      }
      reduce_cols(ctx, part.get(), int(grid), width, sum.get());
      groups.push_back(Group{a0, b0, nta, ntb, ctx.download(sum.get(), width)});
      ctx.keep_until_flush(std::move(part));
      ctx.keep_until_flush(std::move(sum));
    }
  }
  ctx.defer([groups = std::move(groups), pairs, full, want, sink = std::move(sink)]() {
    std::vector<cplx> out(pairs.size());
    for (const Group& gr : groups)
      for (size_t d = 0; d < pairs.size(); d++) {
        const int a = pairs[d].x - gr.a0, b = pairs[d].y - gr.b0;
        if (a < 0 || b < 0 || a >= gr.nta * PM_TILE || b >= gr.ntb * PM_TILE) continue;
        const int tile = a / PM_TILE * gr.ntb + b / PM_TILE;
        const double* h = gr.h + tile * 256 + a % PM_TILE * 16 + b % PM_TILE;
        out[d] = full ? cplx(h[0], h[gr.nta * gr.ntb * 256])
                      : (want == PAIR_IMAG ? cplx(0., h[0]) : cplx(h[0], 0.));
      }
    sink(std::move(out));
  });
}

// pair_reduce of a table on the vector units (k_pair_lds): FP64 fields and two
// real sides.
template <typename T>
static void pair_reduce_lds(Context& ctx, const c2<T>* FA, int na, bool a_packed,
                            const c2<T>* FB, int nbf, bool b_packed, const c2<T>* G,
                            const std::vector<int2>& pairs,
                            std::function<void(std::vector<cplx>&&)> sink) {
  const int mode = (a_packed && b_packed) ? 2 : (b_packed ? 1 : 0);
  const long long nm = ctx.g.nmesh;
  const int rbn = (na + 3) / 4, cbn = (nbf + 3) / 4;
  // Active 4x4 tiles of the (ia, ib) grid.
  std::vector<char> active((size_t)rbn * cbn, 0);
  for (const int2& pr : pairs) active[(size_t)(pr.x / 4) * cbn + pr.y / 4] = 1;
  // Per launch group: its tiles, origin and the host copy of its sums.
  struct Group {
    std::vector<int2> tl;
    int ra0, ca0;
    const double2* h;
  };
  std::vector<Group> groups;
  // Column blocks per launch and row blocks to match: at most 32 fields a
  // side, PT_MAXT tiles and PT_MAXROWS staged rows (4 per block a side).
  const int CB = std::min(cbn, 8);
  const int RB = std::max(1, std::min(std::min((PT_MAXROWS - 1 - 4 * CB) / 4, PT_MAXT / CB), 8));
  // Whole chunks; the kernel reads the cells past the last one directly.
  const long long nchunks = nm / PairLds<T>::LDC;
  for (int c0b = 0; c0b < cbn; c0b += CB) {
    const int c1b = std::min(cbn, c0b + CB);
    for (int r0b = 0; r0b < rbn; r0b += RB) {
      const int r1b = std::min(rbn, r0b + RB);
      std::vector<int2> tl;
      for (int rb = r0b; rb < r1b; rb++)
        for (int cb = c0b; cb < c1b; cb++)
          if (active[(size_t)rb * cbn + cb]) tl.push_back(make_int2(4 * (rb - r0b), 4 * (cb - c0b)));
      if (tl.empty()) continue;
      const int ra0 = 4 * r0b, ca0 = 4 * c0b;
      const int nas = std::min(na, 4 * r1b) - ra0;
      const int nbs = std::min(nbf, 4 * c1b) - ca0;
      const int nt = int(tl.size());
      DevArray<int2> dt(nt);
      ctx.upload(dt.get(), tl.data(), nt);
      // Resident blocks only (each loops over chunks): as many per CU as
      // the double-buffered staging allows.
      const bool same_side = mode == 2 && FA == FB && ra0 == ca0 && nas == nbs;
      const int kmode = same_side ? 3 : mode;
      const size_t smem = pair_lds_smem<T>(kmode, nas, nbs);
      const int per_cu = std::max(1, std::min(8, int((160 * 1024) / smem)));
      const unsigned grid = unsigned(std::min<long long>(nchunks, (long long)ctx.sm_count * per_cu));
      DevArray<double2> part((size_t)grid * nt * 16), sum((size_t)nt * 16);
      {
        // Packed sides start at mesh ra0 / 2 (group starts are multiples of 4).
        const c2<T>* fa = FA + (long long)(mode == 2 ? ra0 / 2 : ra0) * nm;
        const c2<T>* fb = FB + (long long)(mode >= 1 ? ca0 / 2 : ca0) * nm;
        const double ma = pair_rows_a(kmode, nas), mb = pair_rows_b(kmode, nbs);
        ProfScope ps(ctx, KC_PAIR_REDUCE, (ma + mb + 1.) * nm * sizeof(c2<T>));
        switch (kmode) {
          case 3: launch_pair_lds<T, 3>(ctx, grid, smem, fa, nas, fb, nbs, G, nm, dt.get(), nt, part.get()); break;
          case 2: launch_pair_lds<T, 2>(ctx, grid, smem, fa, nas, fb, nbs, G, nm, dt.get(), nt, part.get()); break;
          case 1: if constexpr (sizeof(T) == 8) launch_pair_lds<T, 1>(ctx, grid, smem, fa, nas, fb, nbs, G, nm, dt.get(), nt, part.get()); break;
          default: if constexpr (sizeof(T) == 8) launch_pair_lds<T, 0>(ctx, grid, smem, fa, nas, fb, nbs, G, nm, dt.get(), nt, part.get()); break;
        }
        TRVG_LAUNCH_CHECK();
      }
      reduce_cols(ctx, part.get(), int(grid), nt * 16, sum.get());
      groups.push_back(Group{tl, ra0, ca0, ctx.download(sum.get(), (size_t)nt * 16)});
      ctx.keep_until_flush(std::move(dt));
      ctx.keep_until_flush(std::move(part));
      ctx.keep_until_flush(std::move(sum));
    }
  }
  ctx.defer([groups = std::move(groups), pairs, na, nbf, sink = std::move(sink)]() {
    // Sums for every pair of every active tile, indexed [ia * nbf + ib].
    std::vector<cplx> full((size_t)na * nbf, cplx(0., 0.));
    for (const Group& gr : groups)
      for (size_t t = 0; t < gr.tl.size(); t++)
        for (int i = 0; i < 4; i++)
          for (int j = 0; j < 4; j++) {
            const int a = gr.ra0 + gr.tl[t].x + i, b = gr.ca0 + gr.tl[t].y + j;
            if (a < na && b < nbf) {
              const double2 v = gr.h[t * 16 + i * 4 + j];
              full[(size_t)a * nbf + b] = cplx(v.x, v.y);
            }
          }
    std::vector<cplx> out(pairs.size());
    for (size_t d = 0; d < pairs.size(); d++)
      out[d] = full[(size_t)pairs[d].x * nbf + pairs[d].y];
    sink(std::move(out));
  });
}

template <typename T, int MODE>
static auto pair_list_kernel(int np) {
  switch (np) {
    case 2: return k_pair_list<T, MODE, 2>;
    case 4: return k_pair_list<T, MODE, 4>;
    case 6: return k_pair_list<T, MODE, 6>;
    default: return k_pair_list<T, MODE, 8>;
  }
}

// pair_reduce of a short list (k_pair_list), in equal batches of at most eight
// pairs.
template <typename T>
static void pair_reduce_list(Context& ctx, const c2<T>* FA, bool a_packed, const c2<T>* FB,
                             bool b_packed, const c2<T>* G, const std::vector<int2>& pairs,
                             std::function<void(std::vector<cplx>&&)> sink) {
  const long long nm = ctx.g.nmesh;
  const int np = int(pairs.size());
  const int batches = (np + 7) / 8;
  // Even, so that the two fields of a packed mesh fall into one batch.
  const int per = ((np + batches - 1) / batches + 1) / 2 * 2;
  const int width = batches * per;
  // Four blocks per CU in all: at eight the streams of a large mesh take 5 to
  // 10 % longer.
  const unsigned grid = unsigned(std::min<long long>(
      (nm + 255) / 256, std::max(1, ctx.sm_count * 4 / batches)));
  DevArray<int2> dl(np);
  ctx.upload(dl.get(), pairs.data(), np);
  DevArray<double2> part((size_t)grid * width), sum(width);
  {
    std::set<int> ma, mb;
    for (const int2& q : pairs) {
      ma.insert(a_packed ? q.x / 2 : q.x);
      mb.insert(b_packed ? q.y / 2 : q.y);
    }
    ProfScope ps(ctx, KC_PAIR_REDUCE,
                 double(ma.size() + mb.size() + batches) * double(nm) * sizeof(c2<T>));
    auto kern = pair_list_kernel<T, 2>(per);
      if (!a_packed) kern = b_packed ? pair_list_kernel<T, 1>(per) : pair_list_kernel<T, 0>(per);
    hipLaunchKernelGGL(kern, dim3(batches, grid), dim3(256), 0, ctx.stream, FA, FB, G, nm,
                       dl.get(), np, part.get());
    TRVG_LAUNCH_CHECK();
  }
  reduce_cols(ctx, part.get(), int(grid), width, sum.get());
  const double2* h = ctx.download(sum.get(), width);
  ctx.keep_until_flush(std::move(dl));
  ctx.keep_until_flush(std::move(part));
  ctx.keep_until_flush(std::move(sum));
  ctx.defer([h, np, sink = std::move(sink)]() {
    std::vector<cplx> out(np);
    for (int d = 0; d < np; d++) out[d] = cplx(h[d].x, h[d].y);
    sink(std::move(out));
  });
}

// S_p = sum_x F_a(x) F_b(x) G(x) for pairs p = (a, b) of logical fields,
// handed to `sink` at the next ctx.flush() (the launches are only queued).
// A side / B side packed: real fields stored two per complex mesh (logical
// field 2q + c is component c of mesh q); g_real: G is real.  `want`: what
// the caller uses of S (the rest may come back as zero).
template <typename T>
static void pair_reduce(Context& ctx, const c2<T>* FA, int na, bool a_packed,
                        const c2<T>* FB, int nbf, bool b_packed, const c2<T>* G,
                        bool g_real, PairPart want, const std::vector<int2>& pairs,
                        std::function<void(std::vector<cplx>&&)> sink) {
  if (a_packed && !b_packed) {
    // The product is symmetric in (a, b): put the packed side second.
    std::vector<int2> sw(pairs.size());
    for (size_t d = 0; d < pairs.size(); d++) sw[d] = make_int2(pairs[d].y, pairs[d].x);
    pair_reduce<T>(ctx, FB, nbf, false, FA, na, true, G, g_real, want, sw, std::move(sink));
    return;
  }
  if (a_packed && !g_real)
    throw Error(TRVG_ERR_INTERNAL, "Real shell pairs need a real G field.");
  // Lists with about one pair per field (diagonal, off-diagonal, row) are
  // streamed: they read no mesh twice, and every product is added in FP64.
  // Fuller tables reuse staged rows.  (FP32 lists with a complex side on the
  // matrix cores, 20 diagonal pairs at 256^3: 541 us against 680 streamed, but
  // with 32 cells summed in FP32 where the vector kernel, 778 us, had four.)
  if (!pairs.empty() && int(pairs.size()) <= na + nbf) {
    pair_reduce_list<T>(ctx, FA, a_packed, FB, b_packed, G, pairs, std::move(sink));
    return;
  }
  if constexpr (sizeof(T) == 4) {
    if (!a_packed) {
      pair_reduce_mfma(ctx, FA, na, FB, nbf, b_packed, G, want, pairs, std::move(sink));
      return;
    }
  }
  pair_reduce_lds<T>(ctx, FA, na, a_packed, FB, nbf, b_packed, G, pairs, std::move(sink));
}

struct TwoPt {
  std::vector<int> nmodes;
  std::vector<cplx> pk, sn;
};

// FieldStats::compute_ylm_wgtd_2pt_stats_in_fourier (field.cpp:2511-2703);
// fb_dc is added to fb at k = 0.
template <typename T>
static void twopt_fourier(Context& ctx, const c2<T>* fa, const c2<T>* fb, double fb_dc,
                          cplx sbar, int ell, int m, const trvg_binning& kb, double modes_in_range,
                          std::function<void(TwoPt&&)> sink) {
  const int nb = kb.num_bins;
  std::shared_ptr<const TwoptMapData> map = twopt_map(ctx, kb.bin_edges, nb);
  // Latency-bound (dependent field loads per cell): eight workgroups per CU.
  unsigned grid = grid_for(ctx, ctx.g.nmesh, 8);
  DevArray<unsigned long long> cnt(nb);
  DevArray<double> part((size_t)grid * nb * 4), sum(nb * 4);
  TRVG_HIP(hipMemsetAsync(cnt.get(), 0, nb * 8, ctx.stream));
  // Compulsory reads: both fields at the modes inside the binning range.
  ProfScope ps(ctx, KC_TWOPT, 2. * modes_in_range * sizeof(c2<T>));
  auto kern = ctx.tab.interlace ? k_twopt_fourier<T, 4, true> : k_twopt_fourier<T, 4, false>;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(RED_THREADS),
                     twopt_smem(nb, 4, ctx.g), ctx.stream, fa, fb, ctx.g, ctx.tab,
                     dmk(sbar.real(), sbar.imag()), ell, m, map->view(), nb,
                     cnt.get(), part.get(), fb_dc);
  TRVG_LAUNCH_CHECK();
  reduce_cols(ctx, part.get(), int(grid), nb * 4, sum.get());
  const unsigned long long* hc = ctx.download(cnt.get(), nb);
  const double* hs = ctx.download(sum.get(), (size_t)nb * 4);
  ctx.defer([map]() {});   // keeps the map alive until the launch has run
  ctx.keep_until_flush(std::move(cnt));
  ctx.keep_until_flush(std::move(part));
  ctx.keep_until_flush(std::move(sum));
  ctx.defer([hc, hs, nb, sink = std::move(sink)]() {
    TwoPt r;
    r.nmodes.resize(nb);
    r.pk.resize(nb);
    r.sn.resize(nb);
    for (int b = 0; b < nb; b++) {
      r.nmodes[b] = int(hc[b]);
      if (hc[b] != 0) {
        double n = double(hc[b]);
        r.pk[b] = cplx(hs[4 * b], hs[4 * b + 1]) / n;
        r.sn[b] = cplx(hs[4 * b + 2], hs[4 * b + 3]) / n;
      } else {
        r.pk[b] = 0.;
        r.sn[b] = 0.;
      }
    }
    sink(std::move(r));
  });
}

struct ShotBins3pcf {
  std::vector<int> npairs;
  std::vector<double> r;
  std::vector<cplx> xi;
};

// FieldStats::compute_uncoupled_shotnoise_for_3pcf binning stage
// (field.cpp:3097-3190).
template <typename T>
static ShotBins3pcf shot_bins_3pcf(Context& ctx, const c2<T>* t, int la, int ma,
                                   int lb, int mb, const trvg_binning& rb) {
  const int nb = rb.num_bins;
  DevArray<double> edges(nb + 1);
  TRVG_HIP(hipMemcpyAsync(edges.get(), rb.bin_edges, (nb + 1) * 8,
                          hipMemcpyHostToDevice, ctx.stream));
  unsigned grid = grid_for(ctx, ctx.g.nmesh, 4);
  DevArray<unsigned long long> cnt(nb);
  DevArray<double> part((size_t)grid * nb * 3), sum(nb * 3);
  TRVG_HIP(hipMemsetAsync(cnt.get(), 0, nb * 8, ctx.stream));
  size_t smem = nb * (3 * 8 + 4);
  ProfScope ps(ctx, KC_TWOPT, double(ctx.g.nmesh) * sizeof(c2<T>));
  hipLaunchKernelGGL((k_3pcf_shot_bins<T>), dim3(grid), dim3(RED_THREADS), smem,
                     ctx.stream, t, ctx.g, la, ma, lb, mb, edges.get(), nb,
                     cnt.get(), part.get());
  TRVG_LAUNCH_CHECK();
  reduce_cols(ctx, part.get(), int(grid), nb * 3, sum.get());
  std::vector<unsigned long long> hc(nb);
  std::vector<double> hs(nb * 3);
  TRVG_HIP(hipMemcpyAsync(hc.data(), cnt.get(), nb * 8, hipMemcpyDeviceToHost, ctx.stream));
  TRVG_HIP(hipMemcpyAsync(hs.data(), sum.get(), nb * 24, hipMemcpyDeviceToHost, ctx.stream));
  TRVG_HIP(hipStreamSynchronize(ctx.stream));
  ShotBins3pcf s;
  s.npairs.resize(nb);
  s.r.resize(nb);
  s.xi.resize(nb);
  const double nf = 1 / ctx.g.vol_cell * (((ctx.p.ell1 + ctx.p.ell2) % 2) ? -1. : 1.);
  for (int b = 0; b < nb; b++) {
    s.npairs[b] = int(hc[b]);
    if (hc[b] != 0) {
      double n = double(hc[b]);
      s.r[b] = hs[3 * b] / n;
      s.xi[b] = cplx(hs[3 * b + 1], hs[3 * b + 2]) / n;
      s.xi[b] *= nf / n;
    } else {
      s.r[b] = rb.bin_centres[b];
      s.xi[b] = 0.;
    }
  }
  return s;
}

// S_ij_k for each (k_a, k_b) (field.cpp:3198-3396) from the shot-noise
// field t(x).
// Sorted distinct values (bins of a side).
static std::vector<int> distinct(const std::vector<int>& v) {
  std::vector<int> u(v);
  std::sort(u.begin(), u.end());
  u.erase(std::unique(u.begin(), u.end()), u.end());
  return u;
}

// Distinct bins of each side of a pair list and the pairs re-indexed into
// them: wavenumber lists (k_eff of the bins) for the shot-noise tables.
struct PairBinLists {
  std::vector<double> ka, kb;
  std::vector<int2> pidx;
};
static PairBinLists pair_bin_lists(const std::vector<double>& keff,
                                   const std::vector<int>& ra,
                                   const std::vector<int>& cb) {
  PairBinLists L;
  std::vector<int> ua = distinct(ra), ub = distinct(cb);
  for (int b : ua) L.ka.push_back(keff[b]);
  for (int b : ub) L.kb.push_back(keff[b]);
  L.pidx.resize(ra.size());
  for (size_t d = 0; d < ra.size(); d++)
    L.pidx[d] = make_int2(int(std::lower_bound(ua.begin(), ua.end(), ra[d]) - ua.begin()),
                          int(std::lower_bound(ub.begin(), ub.end(), cb[d]) - ub.begin()));
  return L;
}

// Index of the radial histogram's staged entries by n = a^2 + b^2 + c^2
// (see k_radial_stage / k_radial_gather), built once per device and mesh.
struct RadialIndex {
  DevArray<int> ofs, idx;
  long long nq = 0, nentries = 0;
};

static std::shared_ptr<const RadialIndex> radial_index(Context& ctx) {
  const Geom& g = ctx.g;
  const std::vector<long long> key = {ctx.dev, g.n[0], g.n[1], g.n[2]};
  static std::mutex mu;
  static std::map<std::vector<long long>, std::shared_ptr<const RadialIndex>> cache;
  {
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
  }
  const int h0 = g.n[0] / 2 + 1, h1 = g.n[1] / 2 + 1, h2 = g.n[2] / 2 + 1;
  const bool swap = g.n[0] == g.n[1];
  const long long nrows = swap ? (long long)h0 * (h0 + 1) / 2 : (long long)h0 * h1;
  const long long ne = nrows * h2;
  if (ne >= (1LL << 31))
    throw Error(TRVG_ERR_PARAM, "Mesh too large for the radial histogram index.");
  auto ri = std::make_shared<RadialIndex>();
  ri->nq = (long long)(g.n[0] / 2) * (g.n[0] / 2) + (long long)(g.n[1] / 2) * (g.n[1] / 2) +
           (long long)(g.n[2] / 2) * (g.n[2] / 2) + 1;
  ri->nentries = ne;
  std::vector<long long> rowsq(nrows);
  for (int a = 0; a < h0; a++)
    for (int b = 0; b < (swap ? a + 1 : h1); b++)
      rowsq[swap ? (long long)a * (a + 1) / 2 + b : (long long)a * h1 + b] =
          (long long)a * a + (long long)b * b;
  std::vector<int> ofs(ri->nq + 1, 0), idx(ne);
  for (long long r = 0; r < nrows; r++)
    for (int c = 0; c < h2; c++) ofs[rowsq[r] + (long long)c * c + 1]++;
  for (long long n = 0; n < ri->nq; n++) ofs[n + 1] += ofs[n];
  std::vector<int> cur(ofs.begin(), ofs.end() - 1);
  for (long long r = 0; r < nrows; r++)
    for (int c = 0; c < h2; c++) idx[cur[rowsq[r] + (long long)c * c]++] = int(r * h2 + c);
  ri->ofs.reset(ri->nq + 1);
  ri->idx.reset(ne);
  TRVG_HIP(hipMemcpyAsync(ri->ofs.get(), ofs.data(), (ri->nq + 1) * sizeof(int),
                          hipMemcpyHostToDevice, ctx.stream));
  TRVG_HIP(hipMemcpyAsync(ri->idx.get(), idx.data(), ne * sizeof(int), hipMemcpyHostToDevice,
                          ctx.stream));
  TRVG_HIP(hipStreamSynchronize(ctx.stream));   // the host vectors go out of scope
  std::lock_guard<std::mutex> lk(mu);
  if (cache.size() >= 8) cache.clear();   // bounded; indexes in use stay alive
  cache[key] = ri;
  return ri;
}

template <typename T>
static void shot_pairs_bispec(Context& ctx, const c2<T>* t, int la, int ma, int lb,
                              int mb, const Spline& sa, const Spline& sb,
                              const std::vector<double>& keff, const std::vector<int>& ra,
                              const std::vector<int>& cb,
                              std::function<void(std::vector<cplx>&&)> sink) {
  const int P = int(ra.size());
  const Geom& g = ctx.g;
  const bool cubic = (g.dr[0] == g.dr[1] && g.dr[1] == g.dr[2]);
  if (cubic) {
    long long nq = (long long)(g.n[0] / 2) * (g.n[0] / 2)
                   + (long long)(g.n[1] / 2) * (g.n[1] / 2)
                   + (long long)(g.n[2] / 2) * (g.n[2] / 2) + 1;
    const PairBinLists L = pair_bin_lists(keff, ra, cb);
    const int nka = int(L.ka.size()), nkb = int(L.kb.size());
    const int nch = shot_tab_chunk(nka, nkb);
    const size_t smem = shot_tab_smem(nka, nkb, nch);
    if (smem > 160 * 1024)
      throw Error(TRVG_ERR_PARAM, "Too many wavenumber bins for the shot-noise tables.");
    DevArray<double> dka(nka), dkb(nkb);
    DevArray<int2> dp(P);
    ctx.upload(dka.get(), L.ka.data(), nka);
    ctx.upload(dkb.get(), L.kb.data(), nkb);
    ctx.upload(dp.get(), L.pidx.data(), P);
    const long long nchunks = (nq + nch - 1) / nch;
    const std::shared_ptr<const RadialIndex> ri = radial_index(ctx);
    DevArray<double> Q(2 * nq);
    DevArray<double2> S(ri->nentries);
    DevArray<double2> part((size_t)nchunks * P), res(P);
    {
      // Algorithmic traffic: t read once (the staging and the index are
      // the price of summing without atomics).
      ProfScope ps(ctx, KC_RADIAL, double(g.nmesh) * sizeof(c2<T>));
      hipLaunchKernelGGL((k_radial_stage<T>), dim3(grid_for(ctx, ri->nentries, 8)),
                         dim3(RED_THREADS), 0, ctx.stream, t, g, la, ma, lb, mb, S.get());
      TRVG_LAUNCH_CHECK();
      hipLaunchKernelGGL(k_radial_gather, dim3(grid_for(ctx, nq * RG_LANES, 8)),
                         dim3(RED_THREADS), 0,
                         ctx.stream, S.get(), ri->ofs.get(), ri->idx.get(), nq, Q.get());
      TRVG_LAUNCH_CHECK();
    }
    {
      // The histogram is read once; partials written and reduced once.
      ProfScope ps(ctx, KC_SHOT_PAIRS, double(nq) * 16. + 2. * nchunks * P * 16.);
      hipLaunchKernelGGL(k_shot_pairs_tab, dim3(unsigned(nchunks)), dim3(256), smem,
                         ctx.stream, Q.get(), nq, g.dr[0], sa.dev(), sb.dev(), dka.get(),
                         nka, dkb.get(), nkb, dp.get(), P, nch, g.vol_cell, part.get());
      TRVG_LAUNCH_CHECK();
      reduce_cols(ctx, part.get(), int(nchunks), P, res.get());
    }
    const double2* h = ctx.download(res.get(), P);
    ctx.keep_until_flush(std::move(dka));
    ctx.keep_until_flush(std::move(dkb));
    ctx.keep_until_flush(std::move(dp));
    ctx.keep_until_flush(std::move(Q));
    ctx.keep_until_flush(std::move(S));
    ctx.keep_until_flush(std::move(part));
    ctx.keep_until_flush(std::move(res));
    ctx.defer([h, P, ri, sink = std::move(sink)]() {
      std::vector<cplx> out(P);
      for (int p = 0; p < P; p++) out[p] = cplx(h[p].x, h[p].y);
      sink(std::move(out));
    });
    return;
  }
  std::vector<double> ka(P), kb(P);
  for (int d = 0; d < P; d++) { ka[d] = keff[ra[d]]; kb[d] = keff[cb[d]]; }
  DevArray<double> dka(P), dkb(P);
  ctx.upload(dka.get(), ka.data(), P);
  ctx.upload(dkb.get(), kb.data(), P);
  const int GP = 8;
  unsigned grid = grid_for(ctx, g.nmesh, 4);
  std::vector<const double2*> hs;
  for (int p0 = 0; p0 < P; p0 += GP) {
    int np = std::min(GP, P - p0);
    DevArray<double2> part((size_t)grid * np), sum(np);
    ProfScope ps(ctx, KC_SHOT_PAIRS, double(g.nmesh) * sizeof(c2<T>));
    hipLaunchKernelGGL((k_shot_pairs_direct<T>), dim3(grid), dim3(RED_THREADS), 0,
                       ctx.stream, t, g, la, ma, lb, mb, sa.dev(), sb.dev(),
                       dka.get() + p0, dkb.get() + p0, np, part.get());
    TRVG_LAUNCH_CHECK();
    reduce_cols(ctx, part.get(), int(grid), np, sum.get());
    hs.push_back(ctx.download(sum.get(), np));
    ctx.keep_until_flush(std::move(part));
    ctx.keep_until_flush(std::move(sum));
  }
  ctx.keep_until_flush(std::move(dka));
  ctx.keep_until_flush(std::move(dkb));
  ctx.defer([hs, P, GP, vol = g.vol_cell, sink = std::move(sink)]() {
    std::vector<cplx> out(P);
    for (int p0 = 0, gi = 0; p0 < P; p0 += GP, gi++) {
      const int np = std::min(GP, P - p0);
      for (int q = 0; q < np; q++)
        out[p0 + q] = cplx(hs[gi][q].x, hs[gi][q].y) * vol;
    }
    sink(std::move(out));
  });
}

// S-bar_LM = S-bar_LM[data] + alpha^3 S-bar_LM[randoms] for every (L, M)
// in `keys` (threept.cpp:771-800; with no data catalogue, alpha^3
// S-bar_LM[randoms], threept.cpp:209-237): one pass per catalogue for up to
// SBAR_MAX_KEYS keys, partials downloaded, one synchronisation.  Call with
// no deferred work pending on the context.
static std::map<std::pair<int, int>, cplx> sbar_table(
    Context& ctx, const DeviceCatalogue* d, const DeviceCatalogue& r, double alpha,
    const std::set<std::pair<int, int>>& keys) {
  const std::vector<std::pair<int, int>> kv(keys.begin(), keys.end());
  struct Chunk {
    size_t k0;
    int nk;
    const double2* hd;
    const double2* hr;
    unsigned gd, gr;
  };
  std::vector<Chunk> chunks;
  for (size_t k0 = 0; k0 < kv.size(); k0 += SBAR_MAX_KEYS) {
    SbarKeys sk{};
    sk.n = int(std::min<size_t>(SBAR_MAX_KEYS, kv.size() - k0));
    for (int q = 0; q < sk.n; q++) {
      sk.ell[q] = kv[k0 + q].first;
      sk.m[q] = kv[k0 + q].second;
    }
    Chunk c{k0, sk.n, nullptr, nullptr, 0u, 0u};
    for (int side = d ? 0 : 1; side < 2; side++) {
      const DeviceCatalogue& cat = side == 0 ? *d : r;
      const unsigned grid = grid_for(ctx, cat.n, 4);
      DevArray<double2> part((size_t)grid * sk.n);
      hipLaunchKernelGGL(k_sbar_multi, dim3(grid), dim3(RED_THREADS), 0, ctx.stream,
                         cat.view(), sk, part.get());
      TRVG_LAUNCH_CHECK();
      const double2* h = ctx.download(part.get(), (size_t)grid * sk.n);
      ctx.keep_until_flush(std::move(part));
      if (side == 0) { c.hd = h; c.gd = grid; } else { c.hr = h; c.gr = grid; }
    }
    chunks.push_back(c);
  }
  ctx.flush();
  std::map<std::pair<int, int>, cplx> out;
  for (const Chunk& c : chunks)
    for (int q = 0; q < c.nk; q++) {
      double dx = 0., dy = 0., rx = 0., ry = 0.;
      for (unsigned b = 0; b < c.gd && c.hd; b++) { dx += c.hd[b * c.nk + q].x; dy += c.hd[b * c.nk + q].y; }
      for (unsigned b = 0; b < c.gr; b++) { rx += c.hr[b * c.nk + q].x; ry += c.hr[b * c.nk + q].y; }
      out[kv[c.k0 + q]] = cplx(dx, dy) + std::pow(alpha, 3) * cplx(rx, ry);
    }
  return out;
}

// ---------------------------------------------------------------------------
// Term enumeration shared by the bispectrum and 3PCF drivers
// (threept.cpp:354-419, 1580-1640).
// ---------------------------------------------------------------------------

struct Term {
  int m1, m2, M;
  double coupling, f_mirror, f_mirror_w3j;
};

static std::vector<Term> enumerate_terms(const trvg_params& p, bool survey) {
  std::vector<Term> terms;
  auto inverse = [](const Term& a, int m1, int m2, int M) {
    return a.m1 + m1 == 0 && a.m2 + m2 == 0 && a.M + M == 0;
  };
  for (int m1 = -p.ell1; m1 <= p.ell1; m1++) {
    for (int m2 = -p.ell2; m2 <= p.ell2; m2++) {
      if (survey) {
        bool vanish = true;
        for (int M = -p.ELL; M <= p.ELL; M++)
          if (std::fabs(coupling_3pt(p.ell1, p.ell2, p.ELL, m1, m2, M)) > 1.e-9) {
            vanish = false;
            break;
          }
        if (vanish) continue;
      }
      int Mlo = survey ? -p.ELL : 0, Mhi = survey ? p.ELL : 0;
      for (int M = Mlo; M <= Mhi; M++) {
        bool redundant = false;
        for (auto& t : terms) if (inverse(t, m1, m2, M)) redundant = true;
        if (redundant) continue;
        double c = coupling_3pt(p.ell1, p.ell2, p.ELL, m1, m2, M);
        if (std::fabs(c) < 1.e-9) continue;
        bool zeros = (m1 == 0 && m2 == 0 && M == 0);
        Term t{m1, m2, M, c, zeros ? 0. : ((p.ELL % 2) ? -1. : 1.), zeros ? 0. : 1.};
        terms.push_back(t);
      }
    }
  }
  return terms;
}

static cplx ipow(int n) {
  static const cplx I(0., 1.);
  return std::pow(I, n);  // threept.cpp:271-272
}

// ---------------------------------------------------------------------------
// Shell-field slabs, reused across terms: a slab holds the inverse-
// transformed shell fields of one (l, m) for a set of bins.  B_202 needs the
// (0, 0) side in every term, B_000 / zeta_000 share one slab for both sides.
// ---------------------------------------------------------------------------

template <typename T>
struct ShellSlab {
  int ell = -1, m = 0;
  int n[3] = {0, 0, 0};     // mesh
  std::vector<int> index;   // bin -> field index in `data`, -1 if absent
  int nfields = 0;
  bool packed = false;      // real fields, two per complex mesh
  DevArray<c2<T>> data;
  bool covers(const Geom& g, int l, int mm, const std::vector<int>& bins) const {
    if (ell != l || m != mm || n[0] != g.n[0] || n[1] != g.n[1] || n[2] != g.n[2]) return false;
    for (int b : bins)
      if (b >= int(index.size()) || index[b] < 0) return false;
    return true;
  }
};

// At most `per_mesh` slabs of one mesh are kept, and cells_max complex cells
// over all meshes (the slabs of the pair under way are always held): the smaller
// meshes of some multipoles share the memory that per_mesh slabs of the full
// mesh took.
template <typename T>
class SlabCache {
 public:
  explicit SlabCache(size_t per_mesh = 2, size_t cells_max = SIZE_MAX)
      : per_mesh_(per_mesh), cells_max_(cells_max) {}

  // Returns a slab of (l, m) covering `bins`, building it with
  // make(slab_base, bins) if needed (field q of the slab at
  // slab_base + q * nmesh, or component q % 2 of mesh q / 2 when packed);
  // evicts the least recently used slabs other than `keep` where room is
  // needed.
  template <class Make>
  ShellSlab<T>* get(Context& ctx, int l, int m, const std::vector<int>& bins,
                    int nb, const ShellSlab<T>* keep, bool packed, Make&& make) {
    for (size_t i = 0; i < entries_.size(); i++)
      if (entries_[i]->covers(ctx.g, l, m, bins)) {
        auto e = std::move(entries_[i]);      // move to the back (MRU)
        entries_.erase(entries_.begin() + i);
        entries_.push_back(std::move(e));
        return entries_.back().get();
      }
    const size_t cells =
        size_t(ctx.g.nmesh) * (packed ? (bins.size() + 1) / 2 : bins.size());
    auto e = std::make_unique<ShellSlab<T>>();
    auto here = [&](const ShellSlab<T>& q) {
      return q.n[0] == ctx.g.n[0] && q.n[1] == ctx.g.n[1] && q.n[2] == ctx.g.n[2];
    };
    size_t same = 0, held = cells;
    for (const auto& q : entries_) {
      same += here(*q);
      held += q->data.size();
    }
    for (size_t i = 0; i < entries_.size();) {
      ShellSlab<T>& q = *entries_[i];
      const bool full = same >= per_mesh_ && here(q);
      if (&q == keep || !(full || held > cells_max_)) {
        i++;
        continue;
      }
      same -= here(q);
      held -= q.data.size();
      // The kernels that read it are still queued: the new slab takes its place
      // in stream order, or it goes back to the shared pool once they are done.
      if (!e->data.get() && q.data.size() == cells) e->data = std::move(q.data);
      else TRVG_HIP(hipStreamSynchronize(ctx.stream));
      entries_.erase(entries_.begin() + i);
    }
    e->ell = l;
    e->m = m;
    for (int a = 0; a < 3; a++) e->n[a] = ctx.g.n[a];
    e->index.assign(nb, -1);
    e->nfields = int(bins.size());
    e->packed = packed;
    if (!e->data.get()) e->data.reset(cells);
    make(e->data.get(), bins);
    for (size_t q = 0; q < bins.size(); q++) e->index[bins[q]] = int(q);
    entries_.push_back(std::move(e));
    return entries_.back().get();
  }

 private:
  size_t per_mesh_, cells_max_;
  std::vector<std::unique_ptr<ShellSlab<T>>> entries_;
};

// ---------------------------------------------------------------------------
// Bispectrum
// ---------------------------------------------------------------------------

SurveyPrefill prefill_survey_data(Context& ctx, const DeviceCatalogue& d,
                                  const std::vector<Multipole>& mps) {
  SurveyPrefill pre;
  if (!std::isfinite(d.wuni)) return pre;
  // Keys in the order the estimator uses them: the common (0, 0) pair, then
  // the (L, M) of each term that is not (0, 0).
  std::vector<std::pair<int, int>> keys{{0, 0}};
  for (const Multipole& mp : mps) {
    trvg_params p = ctx.p;
    p.ell1 = mp.ell1; p.ell2 = mp.ell2; p.ELL = mp.ELL;
    for (const Term& tm : enumerate_terms(p, true))
      if (!(p.ELL == 0 && tm.M == 0)) keys.push_back({p.ELL, tm.M});
  }
  constexpr size_t cap = size_t(4) << 30;
  const size_t bytes = size_t(ctx.g.nmesh) * sizeof(double2);
  size_t held = 0;
  for (const auto& k : keys) {
    if (pre.sd.count(k)) continue;
    if (held + bytes > cap) break;
    held += bytes;
    // As build_survey_pair_k assigns the data side of a uniform pair.
    DevArray<double2> f(ctx.g.nmesh);
    zero_field<double>(ctx, f.get());
    assign<double>(ctx, f.get(), d, WM_YLM_W, k.first, k.second, 1.);
    pre.sd.emplace(k, std::move(f));
  }
  return pre;
}

template <typename T>
std::vector<Result> run_bispec_multi(Context& ctx, const DeviceCatalogue& d,
                                     const DeviceCatalogue* r, bool survey,
                                     const trvg_binning& kb,
                                     const std::vector<Multipole>& mps,
                                     SurveyPrefill* pre) {
  const Geom g = ctx.g;   // a copy: the pair sums may run on another mesh
  const long long nm = g.nmesh;
  const double alpha = survey ? d.wstotal / r->wstotal : 1.;
  const int nb = kb.num_bins;

  // S_d of (L, M) assigned ahead of the random catalogue (uniform weights
  // on both sides only), taken once; an empty array when there is none.
  const bool uniform = survey && std::isfinite(d.wuni) && std::isfinite(r->wuni);
  auto take_prefill = [&](int L, int M) {
    DevArray<double2> f;
    if (pre && uniform) {
      auto it = pre->sd.find({L, M});
      if (it != pre->sd.end()) {
        f = std::move(it->second);
        pre->sd.erase(it);
      }
    }
    return f;
  };

  // Common fields in FP64 whatever the shell precision T: the shot-noise
  // path (two-point statistics, S_ij_k) subtracts nearly equal quantities.
  DevArray<double2> dn00 = take_prefill(0, 0), N00(survey ? nm : 0);
  const bool dn00_pre = dn00.get() != nullptr;
  if (!dn00_pre) dn00.reset(nm);
  if (survey) {
    build_survey_pair_k(ctx, dn00.get(), N00.get(), d, *r, alpha, 0, 0, dn00_pre);
  } else {
    build_field_k<double>(ctx, dn00.get(), d, r, false, alpha, 0, 0, false, true);
  }
  // A box has unit weights: N_00 is the density itself, dn_00 with the mean
  // (the particle count) back at k = 0, so it is neither assigned nor
  // transformed.
  const double2* N00p = survey ? N00.get() : dn00.get();
  const double N_dc = survey ? 0. : double(d.n);
  ShellStats ss = shell_stats(ctx, kb);
  double modes_in_range = 0.;
  for (int n : ss.nmodes) modes_in_range += n;

  auto spline = [&](int ell) -> const Spline& {
    return cached_spline(ctx.dev, ell, ctx.stream);
  };

  DevArray<c2<T>> G(nm);
  // t(x) in the working precision (an FP32 transform in the FP32 path; its
  // radial histogram and the pair sums over it accumulate in FP64).
  DevArray<c2<T>> tfield(nm);
  DevArray<double2> dnLM, NLM;
  // Inputs of the shot-noise field held in tfield: (L, M) of its dn field
  // (-1 for dn00) and Sbar; a periodic box uses one t(x) for every term and
  // multipole.
  int t_ell = -2, t_m = 0;
  cplx t_sbar(0., 0.);
  // Meshes of each multipole's pair sums, and dn00(k) / W(k) on them.
  std::vector<std::vector<MeshGroup>> plans;
  long long nm_coarse = 0;
  size_t slab_max = 0;   // cells of the largest slab that the full mesh would take
  for (const Multipole& mp : mps) {
    std::vector<int> ra, cb;
    pair_bins(mp.shape, nb, mp.idx_bin, ra, cb);
    const bool split = mp.shape != TRVG_SHAPE_FULL && mp.shape != TRVG_SHAPE_TRIU;
    plans.push_back(plan_mesh_groups(g, kb, ra, cb, split, sizeof(c2<T>)));
    for (const MeshGroup& gr : plans.back())
      if (gr.coarse) nm_coarse = std::max(nm_coarse, mesh_of(g, gr.n).nmesh);
    trvg_params p = ctx.p;
    p.ell1 = mp.ell1; p.ell2 = mp.ell2; p.ELL = mp.ELL;
    auto cells = [&](int l, int m, size_t fields) {
      return size_t(nm) * (real_shells(l, m) ? (fields + 1) / 2 : fields);
    };
    for (const Term& tm : enumerate_terms(p, survey)) {
      slab_max = std::max(slab_max, cells(p.ell1, tm.m1, distinct(ra).size()));
      slab_max = std::max(slab_max, cells(p.ell2, tm.m2, distinct(cb).size()));
    }
  }
  std::map<std::vector<int>, DevArray<double2>> coarse00;
  DevArray<double2> coarseLM;
  const size_t per_mesh = mps.size() > 1 ? 3 : 2;
  SlabCache<T> slabs(per_mesh, per_mesh * slab_max);
  auto make_shell = [&](const double2* src, int l, int mm) {
    return [&, src, l, mm](c2<T>* base, const std::vector<int>& bins) {
      shell_slab_ifft<T, double>(ctx, base, src, kb, bins, ss.nmodes, l, mm, real_shells(l, mm));
    };
  };

  // S-bar_LM of every term of every multipole, computed up front.
  std::map<std::pair<int, int>, cplx> sbar;
  if (survey) {
    std::set<std::pair<int, int>> keys;
    for (const Multipole& mp : mps) {
      trvg_params p = ctx.p;
      p.ell1 = mp.ell1; p.ell2 = mp.ell2; p.ELL = mp.ELL;
      for (const Term& tm : enumerate_terms(p, survey)) keys.insert({p.ELL, tm.M});
    }
    sbar = sbar_table(ctx, &d, *r, alpha, keys);
  }

  std::vector<Result> results;
  for (const Multipole& mp : mps) {
    trvg_params p = ctx.p;
    p.ell1 = mp.ell1; p.ell2 = mp.ell2; p.ELL = mp.ELL;
    p.shape = mp.shape; p.idx_bin = mp.idx_bin;
    const cplx factor_phase = ipow(p.ell1 + p.ell2);
    std::vector<int> ra, cb;
    pair_bins(p.shape, nb, p.idx_bin, ra, cb);
    const int dim = int(ra.size());
    const std::vector<MeshGroup>& plan = plans[results.size()];

    Result out;
    out.dim = dim;
    out.b1.resize(dim); out.b2.resize(dim); out.e1.resize(dim); out.e2.resize(dim);
    out.n1.resize(dim); out.n2.resize(dim);
    out.raw.assign(dim, 0.); out.shot.assign(dim, 0.);
    for (int dv = 0; dv < dim; dv++) {
      out.b1[dv] = kb.bin_centres[ra[dv]];
      out.b2[dv] = kb.bin_centres[cb[dv]];
      out.e1[dv] = ss.keff[ra[dv]];
      out.e2[dv] = ss.keff[cb[dv]];
      out.n1[dv] = ss.nmodes[ra[dv]];
      out.n2[dv] = ss.nmodes[cb[dv]];
    }
    const Spline& sja = spline(p.ell1);
    const Spline& sjb = spline(p.ell2);

    for (const Term& tm : enumerate_terms(p, survey)) {
      const bool lm_zero = !survey || (p.ELL == 0 && tm.M == 0);
      const double2* dnLMp = dn00.get();
      const double2* NLMp = N00p;
      if (!lm_zero) {
        if (!NLM.get()) NLM.reset(nm);
        DevArray<double2> own = take_prefill(p.ELL, tm.M);
        if (own.get()) {
          build_survey_pair_k(ctx, own.get(), NLM.get(), d, *r, alpha, p.ELL, tm.M, true);
          dnLMp = own.get();
          ctx.keep_until_flush(std::move(own));   // read by this term's kernels
        } else {
          if (!dnLM.get()) dnLM.reset(nm);
          build_survey_pair_k(ctx, dnLM.get(), NLM.get(), d, *r, alpha, p.ELL, tm.M);
          dnLMp = dnLM.get();
        }
        NLMp = NLM.get();
      }

      // G_LM is real for M = 0 (real weights Y_L0) and in a periodic box.
      const bool g_real = !survey || tm.M == 0;
      const double coupling = tm.coupling, f_mirror = tm.f_mirror;
      for (const MeshGroup& gr : plan) {
        const double2 *src00 = dn00.get(), *srcLM = dnLMp;
        const Geom gc = gr.coarse ? mesh_of(g, gr.n) : g;
        if (gr.coarse) {
          DevArray<double2>& c00 = coarse00[{gr.n[0], gr.n[1], gr.n[2]}];
          if (!c00.get()) {
            c00.reset(gc.nmesh);
            truncate_modes<double>(ctx, dn00.get(), gc, c00.get());
          }
          src00 = srcLM = c00.get();
          if (dnLMp != dn00.get()) {
            if (!coarseLM.get()) coarseLM.reset(nm_coarse);
            truncate_modes<double>(ctx, dnLMp, gc, coarseLM.get());
            srcLM = coarseLM.get();
          }
        }
        std::unique_ptr<MeshScope> scope;
        if (gr.coarse) scope = std::make_unique<MeshScope>(ctx, gc);
        std::vector<int> gra, gcb;
        for (int dv : gr.pairs) { gra.push_back(ra[dv]); gcb.push_back(cb[dv]); }
        const std::vector<int> rows = distinct(gra), cols = distinct(gcb);

        // G_LM(x): compensated, inverse-transformed (threept.cpp:452-459).
        LoadDeconv<T, double> ldg{srcLM, ctx.tab, 1. / g.vol};
        fft3d<T>(ctx, G.get(), ldg, +1, double(gc.nmesh) * sizeof(double2));

        // Shell fields F_a (l1, m1) for the row bins, F_b (l2, m2) for columns.
        ShellSlab<T>* A =
            slabs.get(ctx, p.ell1, tm.m1, rows, nb, nullptr, real_shells(p.ell1, tm.m1),
                      make_shell(src00, p.ell1, tm.m1));
        ShellSlab<T>* B =
            slabs.get(ctx, p.ell2, tm.m2, cols, nb, A, real_shells(p.ell2, tm.m2),
                      make_shell(src00, p.ell2, tm.m2));
        std::vector<int2> pairs(gra.size());
        for (size_t d = 0; d < gra.size(); d++)
          pairs[d] = make_int2(A->index[gra[d]], B->index[gcb[d]]);
        // Results arrive at the flush after the last term (the sinks add
        // into `out`, which outlives them).
        pair_reduce<T>(ctx, A->data.get(), A->nfields, A->packed, B->data.get(),
                       B->nfields, B->packed, G.get(), g_real, wanted(f_mirror), pairs,
                       [&out, &ra, &cb, &ss, dvs = gr.pairs, coupling, f_mirror,
                        vc = gc.vol_cell](std::vector<cplx>&& S) {
                         for (size_t d = 0; d < dvs.size(); d++) {
                           const int dv = dvs[d];
                           cplx sv = S[d] / (double(ss.nmodes[ra[dv]]) *
                                             double(ss.nmodes[cb[dv]]));
                           out.raw[dv] += coupling * vc * (sv + f_mirror * std::conj(sv));
                         }
                       });
      }

      // Shot noise (threept.cpp:771-966).
      const cplx Sbar = survey ? sbar.at({p.ELL, tm.M}) : cplx(double(d.n), 0.);
      if (p.ell1 == 0 && p.ell2 == 0) {
        cplx sijk = tm.coupling * Sbar;
        for (int dv = 0; dv < dim; dv++) out.shot[dv] += sijk;
      }
      // Two-point terms of the row side (ell2 = 0) and/or the column side
      // (ell1 = 0); with both sides monopoles of one m the statistics are
      // shared.
      auto twopt_sink = [&out, &ra, &cb, dim, coupling, f_mirror](bool rows, bool cols) {
        return [&out, &ra, &cb, dim, coupling, f_mirror, rows, cols](TwoPt&& st) {
          for (int side = 0; side < 2; side++) {
            if (!(side == 0 ? rows : cols)) continue;
            const std::vector<int>& bins = side == 0 ? ra : cb;
            for (int dv = 0; dv < dim; dv++) {
              int bb = bins[dv];
              cplx sv = coupling * (st.pk[bb] - st.sn[bb]);
              out.shot[dv] += sv + f_mirror * std::conj(sv);
            }
          }
        };
      };
      const bool shared = p.ell1 == 0 && p.ell2 == 0 && tm.m1 == tm.m2;
      if (p.ell2 == 0)
        twopt_fourier<double>(ctx, dn00.get(), NLMp, N_dc, Sbar, p.ell1, tm.m1, kb,
                              modes_in_range, twopt_sink(true, shared));
      if (p.ell1 == 0 && !shared)
        twopt_fourier<double>(ctx, dn00.get(), NLMp, N_dc, Sbar, p.ell2, tm.m2, kb,
                              modes_in_range, twopt_sink(false, true));
      const int key_ell = lm_zero ? -1 : p.ELL, key_m = lm_zero ? 0 : tm.M;
      if (key_ell != t_ell || key_m != t_m || Sbar != t_sbar) {
        LoadTwopt<T, double> lt{dnLMp, N00p, ctx.tab, dmk(Sbar.real(), Sbar.imag()),
                                1. / g.vol, N_dc};
        fft3d<T>(ctx, tfield.get(), lt, +1, 2. * double(nm) * sizeof(double2));
        t_ell = key_ell;
        t_m = key_m;
        t_sbar = Sbar;
      }
      shot_pairs_bispec<T>(
          ctx, tfield.get(), p.ell1, tm.m1, p.ell2, tm.m2, sja, sjb, ss.keff, ra, cb,
          [&out, dim, coupling, factor_phase, fmw = tm.f_mirror_w3j](std::vector<cplx>&& sij) {
            for (int dv = 0; dv < dim; dv++) {
              cplx sv = coupling * sij[dv];
              out.shot[dv] += factor_phase * (sv + fmw * std::conj(sv));
            }
          });
    }
    ctx.flush();
    for (int dv = 0; dv < dim; dv++) {
      out.raw[dv] *= mp.norm;
      out.shot[dv] *= mp.norm;
    }
    results.push_back(std::move(out));
  }
  return results;
}

template <typename T>
Result run_bispec(Context& ctx, const DeviceCatalogue& d,
                  const DeviceCatalogue* r, bool survey,
                  const trvg_binning& kb, double norm_factor, SurveyPrefill* pre) {
  Multipole mp{ctx.p.ell1, ctx.p.ell2, ctx.p.ELL, ctx.p.shape, ctx.p.idx_bin,
               norm_factor};
  return std::move(run_bispec_multi<T>(ctx, d, r, survey, kb, {mp}, pre)[0]);
}

// ---------------------------------------------------------------------------
// Three-point correlation function
// ---------------------------------------------------------------------------

template <typename T>
Result run_3pcf(Context& ctx, const DeviceCatalogue& d,
                const DeviceCatalogue* r, bool survey,
                const trvg_binning& rb, double norm_factor,
                const Window3pcf* win) {
  const trvg_params& p = ctx.p;
  const Geom& g = ctx.g;
  const long long nm = g.nmesh;
  const double alpha = win ? win->alpha : (survey ? d.wstotal / r->wstotal : 1.);
  const cplx factor_phase = ipow(p.ell1 + p.ell2);
  const double factor_parity = ((p.ell1 + p.ell2) % 2) ? -1. : 1.;
  const int nb = rb.num_bins;
  std::vector<int> ra, cb;
  pair_bins(p.shape, nb, p.idx_bin, ra, cb);
  const int dim = int(ra.size());

  Result out;
  out.dim = dim;
  out.b1.resize(dim); out.b2.resize(dim); out.e1.resize(dim); out.e2.resize(dim);
  out.n1.resize(dim); out.n2.resize(dim);
  out.raw.assign(dim, 0.); out.shot.assign(dim, 0.);

  DevArray<double2> dn00(nm), N00(survey ? nm : 0);
  if (win) {
    build_single_field_k(ctx, dn00.get(), d, alpha, 0, 0, false);
    build_single_field_k(ctx, N00.get(), d, alpha, 0, 0, true);
  } else if (survey) {
    build_survey_pair_k(ctx, dn00.get(), N00.get(), d, *r, alpha, 0, 0);
  } else {
    build_field_k<double>(ctx, dn00.get(), d, r, false, alpha, 0, 0, false, true);
  }
  // N_00 of a box from dn_00, as in run_bispec_multi.
  const double2* N00p = survey ? N00.get() : dn00.get();
  const double N_dc = survey ? 0. : double(d.n);

  const Spline& sja = cached_spline(ctx.dev, p.ell1, ctx.stream);
  const Spline& sjb = cached_spline(ctx.dev, p.ell2, ctx.stream);

  std::vector<int> rows = distinct(ra), cols = distinct(cb);
  DevArray<c2<T>> G(nm);
  DevArray<c2<T>> tfield(nm);
  DevArray<double2> dnLM;
  SlabCache<T> slabs;
  std::vector<double> reff(nb, 0.);
  bool first = true;
  std::map<std::pair<int, int>, cplx> sbar;
  if (survey) {
    std::set<std::pair<int, int>> keys;
    for (const Term& tm : enumerate_terms(p, survey)) keys.insert({p.ELL, tm.M});
    sbar = win ? sbar_table(ctx, nullptr, d, alpha, keys)
               : sbar_table(ctx, &d, *r, alpha, keys);
  }

  for (const Term& tm : enumerate_terms(p, survey)) {
    const bool lm_zero = !survey || (p.ELL == 0 && tm.M == 0);
    const double2* dnLMp = dn00.get();
    if (!lm_zero) {
      if (!dnLM.get()) dnLM.reset(nm);
      if (win)
        build_single_field_k(ctx, dnLM.get(), d, alpha, p.ELL, tm.M, false);
      else
        build_field_k<double>(ctx, dnLM.get(), d, r, true, alpha, p.ELL, tm.M, false, false);
      dnLMp = dnLM.get();
    }
    const cplx Sbar = survey ? sbar.at({p.ELL, tm.M}) : cplx(double(d.n), 0.);

    // Shot noise first: defines r_eff and n_pairs (threept.cpp:1223-1367).
    LoadTwopt<T, double> lt{dnLMp, N00p, ctx.tab, dmk(Sbar.real(), Sbar.imag()),
                            1. / g.vol, N_dc};
    fft3d<T>(ctx, tfield.get(), lt, +1, 2. * double(nm) * sizeof(double2));
    ShotBins3pcf sb = shot_bins_3pcf<T>(ctx, tfield.get(), p.ell1, tm.m1, p.ell2,
                                        tm.m2, rb);
    for (int dv = 0; dv < dim; dv++) {
      if (ra[dv] != cb[dv]) continue;
      if (p.shape == TRVG_SHAPE_OFFDIAG && p.idx_bin != 0) continue;
      int b = ra[dv];
      out.shot[dv] += tm.coupling * factor_parity
                      * (sb.xi[b] + tm.f_mirror_w3j * std::conj(sb.xi[b]));
    }
    if (first) {
      for (int dv = 0; dv < dim; dv++) {
        out.b1[dv] = rb.bin_centres[ra[dv]];
        out.b2[dv] = rb.bin_centres[cb[dv]];
        out.e1[dv] = sb.r[ra[dv]];
        out.e2[dv] = sb.r[cb[dv]];
        out.n1[dv] = sb.npairs[ra[dv]];
        out.n2[dv] = sb.npairs[cb[dv]];
      }
      reff = sb.r;
      first = false;
    }

    LoadDeconv<T, double> ldg{dnLMp, ctx.tab, 1. / g.vol};
    fft3d<T>(ctx, G.get(), ldg, +1, double(nm) * sizeof(double2));
    if (win && win->wa_power >= 0) {
      // Wide-angle power-law kernel (field.cpp:1727-1762).
      ProfScope ps(ctx, KC_MISC, 2. * double(nm) * sizeof(c2<T>));
      hipLaunchKernelGGL((k_wide_angle<T>), dim3(grid_for(ctx, nm)), dim3(RED_THREADS), 0,
                         ctx.stream, G.get(), g, win->wa_power);
      TRVG_LAUNCH_CHECK();
    }

    auto make_sjl = [&](int l, int mm, const Spline& sp) {
      return [&, l, mm](c2<T>* base, const std::vector<int>& bins) {
        sjl_slab_ifft<T>(ctx, base, dn00.get(), sp, reff, bins, l, mm, real_shells(l, mm));
      };
    };
    ShellSlab<T>* A = slabs.get(ctx, p.ell1, tm.m1, rows, nb, nullptr,
                                real_shells(p.ell1, tm.m1), make_sjl(p.ell1, tm.m1, sja));
    ShellSlab<T>* B = slabs.get(ctx, p.ell2, tm.m2, cols, nb, A,
                                real_shells(p.ell2, tm.m2), make_sjl(p.ell2, tm.m2, sjb));
    std::vector<int2> pairs(dim);
    for (int dv = 0; dv < dim; dv++)
      pairs[dv] = make_int2(A->index[ra[dv]], B->index[cb[dv]]);
    // G_LM is real for M = 0 (real weights Y_L0) and in a periodic box.
    const bool g_real = !survey || tm.M == 0;
    pair_reduce<T>(ctx, A->data.get(), A->nfields, A->packed, B->data.get(), B->nfields,
                   B->packed, G.get(), g_real, wanted(tm.f_mirror), pairs,
                   [&out, dim, c = tm.coupling * g.vol_cell * factor_phase,
                    fm = tm.f_mirror](std::vector<cplx>&& S) {
                     for (int dv = 0; dv < dim; dv++)
                       out.raw[dv] += c * (S[dv] + fm * std::conj(S[dv]));
                   });
  }
  ctx.flush();
  for (int dv = 0; dv < dim; dv++) {
    out.raw[dv] *= norm_factor;
    out.shot[dv] *= norm_factor;
  }
  return out;
}

// calc_bispec_normalisation_from_mesh (threept.cpp:138-149 ->
// field.cpp:2017-2065) before the 1/alpha^3 factor.
template <typename T>
double run_mesh_norm(Context& ctx, const DeviceCatalogue& c) {
  // A single assignment and reduction: always FP64.
  DevArray<double2> f(ctx.g.nmesh);
  zero_field<double>(ctx, f.get());
  assign<double>(ctx, f.get(), c, WM_W, 0, 0, 1.);
  unsigned grid = grid_for(ctx, ctx.g.nmesh, 4);
  DevArray<double> part(grid), sum(1);
  hipLaunchKernelGGL((k_cube_sum<double>), dim3(grid), dim3(RED_THREADS), 0,
                     ctx.stream, f.get(), ctx.g.nmesh, part.get());
  TRVG_LAUNCH_CHECK();
  reduce_cols(ctx, part.get(), int(grid), 1, sum.get());
  double h = 0.;
  TRVG_HIP(hipMemcpyAsync(&h, sum.get(), 8, hipMemcpyDeviceToHost, ctx.stream));
  TRVG_HIP(hipStreamSynchronize(ctx.stream));
  return 1. / (h * ctx.g.vol_cell);
}

template std::vector<Result> run_bispec_multi<double>(
    Context&, const DeviceCatalogue&, const DeviceCatalogue*, bool,
    const trvg_binning&, const std::vector<Multipole>&, SurveyPrefill*);
template std::vector<Result> run_bispec_multi<float>(
    Context&, const DeviceCatalogue&, const DeviceCatalogue*, bool,
    const trvg_binning&, const std::vector<Multipole>&, SurveyPrefill*);
template Result run_bispec<double>(Context&, const DeviceCatalogue&,
                                   const DeviceCatalogue*, bool,
                                   const trvg_binning&, double, SurveyPrefill*);
template Result run_bispec<float>(Context&, const DeviceCatalogue&,
                                  const DeviceCatalogue*, bool,
                                  const trvg_binning&, double, SurveyPrefill*);
template Result run_3pcf<double>(Context&, const DeviceCatalogue&,
                                 const DeviceCatalogue*, bool,
                                 const trvg_binning&, double, const Window3pcf*);
template Result run_3pcf<float>(Context&, const DeviceCatalogue&,
                                const DeviceCatalogue*, bool,
                                const trvg_binning&, double, const Window3pcf*);
template double run_mesh_norm<double>(Context&, const DeviceCatalogue&);
template double run_mesh_norm<float>(Context&, const DeviceCatalogue&);

}  // namespace trvg

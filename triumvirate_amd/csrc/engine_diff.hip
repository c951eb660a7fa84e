// engine_diff.hip -- differentiable periodic-box bispectrum B_000 (diag
// form) and mesh assignment: forward, hand-written adjoints, C ABI.
//
// The forward is the chain of compute_bispec_in_gpp_box (threept.cpp:
// 1473-2188) for l1 = l2 = L = 0 with the diag form, starting from a given
// real mesh delta(x) (the unweighted field fluctuation of
// field.cpp:1235-1243 when delta comes from trvg_diff_assign minus the
// mean).  Shell fields are recomputed in the backward pass instead of being
// stored.  Bins whose products fit a smaller mesh run there (MeshGroup), two
// real shells per transform.  Device pointers in, host vectors of per-bin
// values out.
#include <cmath>
#include <vector>

#include "diff_kernels.hpp"
#include "engine.hpp"

namespace trvg {

namespace {

// The bins that share one mesh (every bin pairs with itself only) and their
// fields there: G(x) and the real shell fields F_b, two per complex mesh
// (bin bins[2p + c] is component c of mesh p).  The slab has one more mesh,
// for the cotangent of G in the backward pass.
template <typename T>
struct DiffGroup {
  std::vector<int> bins;
  Geom g;
  bool coarse;
  int nt;
  DevArray<c2<T>> D, G, F;
};

// D(k) of the mesh, then per group of `bins` G and the shells.
template <typename T>
std::vector<DiffGroup<T>> diff_groups(Context& ctx, const trvg_binning& kb, const T* mesh,
                                      const std::vector<int>& nmodes,
                                      const std::vector<int>& bins) {
  const Geom g = ctx.g;
  DevArray<c2<T>> D(g.nmesh);
  fft3d<T>(ctx, D.get(), LoadReal<T>{mesh, T(g.vol_cell)}, -1, double(g.nmesh) * sizeof(T));
  std::vector<DiffGroup<T>> out;
  for (const MeshGroup& gr : plan_mesh_groups(g, kb, bins, bins, true, sizeof(c2<T>))) {
    DiffGroup<T> d;
    for (int q : gr.pairs) d.bins.push_back(bins[q]);   // a bin pairs with itself
    d.coarse = gr.coarse;
    d.g = gr.coarse ? mesh_of(g, gr.n) : g;
    d.nt = (int(d.bins.size()) + 1) / 2;
    const c2<T>* src = D.get();
    if (gr.coarse) {
      d.D.reset(d.g.nmesh);
      truncate_modes<T>(ctx, D.get(), d.g, d.D.get());
      src = d.D.get();
    }
    std::unique_ptr<MeshScope> scope;
    if (gr.coarse) scope = std::make_unique<MeshScope>(ctx, d.g);
    d.G.reset(d.g.nmesh);
    fft3d<T>(ctx, d.G.get(), LoadDeconv<T, T>{src, ctx.tab, 1. / g.vol}, +1);
    d.F.reset(size_t(d.nt + 1) * d.g.nmesh);
    shell_slab_ifft<T, T>(ctx, d.F.get(), src, kb, d.bins, nmodes, 0, 0, true);
    out.push_back(std::move(d));
  }
  ctx.keep_until_flush(std::move(D));
  return out;
}

}  // namespace

template <typename T>
std::vector<double> diff_bispec_forward(Context& ctx, const trvg_binning& kb,
                                        double norm, const T* mesh,
                                        std::vector<int>& nmodes) {
  ShellStats ss = shell_stats(ctx, kb);
  nmodes = ss.nmodes;
  std::vector<int> bins(kb.num_bins);
  for (int b = 0; b < kb.num_bins; b++) bins[b] = b;
  std::vector<DiffGroup<T>> groups = diff_groups<T>(ctx, kb, mesh, ss.nmodes, bins);
  std::vector<const double*> h;
  for (DiffGroup<T>& d : groups) {
    const int nv = 2 * d.nt;
    const unsigned grid = grid_for(ctx, d.g.nmesh, 4);
    DevArray<double> part((size_t)grid * nv), sums(nv);   // [grid][nv]
    ProfScope ps(ctx, KC_PAIR_REDUCE, double(d.nt + 1) * double(d.g.nmesh) * sizeof(c2<T>));
    hipLaunchKernelGGL((k_f2g_packed<T>), dim3(grid, unsigned(d.nt)), dim3(RED_THREADS), 0,
                       ctx.stream, d.F.get(), d.G.get(), d.g.nmesh, part.get());
    TRVG_LAUNCH_CHECK();
    reduce_cols(ctx, part.get(), int(grid), nv, sums.get());
    h.push_back(ctx.download(sums.get(), nv));
    ctx.keep_until_flush(std::move(part));
    ctx.keep_until_flush(std::move(sums));
  }
  ctx.flush();
  std::vector<double> out(kb.num_bins);
  for (size_t q = 0; q < groups.size(); q++)
    for (size_t i = 0; i < groups[q].bins.size(); i++) {
      const int b = groups[q].bins[i];
      const double n = double(ss.nmodes[b]);
      out[b] = norm * groups[q].g.vol_cell * h[q][i] / (n * n);   // NaN for an empty bin
    }
  return out;
}

template <typename T>
void diff_bispec_backward(Context& ctx, const trvg_binning& kb, double norm,
                          const T* mesh, const double* grad_bk, T* grad_mesh) {
  const Geom g = ctx.g;
  const long long nm = g.nmesh;
  const int nb = kb.num_bins;
  ShellStats ss = shell_stats(ctx, kb);
  // Bins that contribute: none costs transforms, or spreads a mesh's infinities
  // and NaN, without a cotangent.
  std::vector<int> bins;
  for (int b = 0; b < nb; b++)
    if (grad_bk[b] != 0. && ss.nmodes[b] != 0) bins.push_back(b);
  std::vector<DiffGroup<T>> groups = diff_groups<T>(ctx, kb, mesh, ss.nmodes, bins);
  DevArray<c2<T>> acc(nm);
  const unsigned grid = grid_for(ctx, nm);
  hipLaunchKernelGGL((k_zero<T>), dim3(grid), dim3(RED_THREADS), 0, ctx.stream,
                     acc.get(), nm);
  TRVG_LAUNCH_CHECK();
  // Thresholds of |k|^2 between the bins (bin b: [edge[b], edge[b + 1])).
  std::vector<double> edge(nb + 1);
  for (int b = 0; b <= nb; b++) edge[b] = sq_threshold(kb.bin_edges[b]);
  DevArray<double> dedge(nb + 1);
  ctx.upload(dedge.get(), edge.data(), nb + 1);
  bool all_coarse = true;
  for (DiffGroup<T>& d : groups) {
    all_coarse = all_coarse && d.coarse;
    std::vector<double> a(2 * d.nt, 0.);
    std::vector<int> slot(nb, -1);
    for (size_t i = 0; i < d.bins.size(); i++) {
      const int b = d.bins[i];
      const double n = double(ss.nmodes[b]);
      a[i] = grad_bk[b] * norm * d.g.vol_cell / (n * n);
      slot[b] = int(i);
    }
    DevArray<double> da(a.size());
    DevArray<int> dslot(nb);
    ctx.upload(da.get(), a.data(), a.size());
    ctx.upload(dslot.get(), slot.data(), nb);
    {
      ProfScope ps(ctx, KC_MISC, (2. * d.nt + 2.) * double(d.g.nmesh) * sizeof(c2<T>));
      hipLaunchKernelGGL((k_cotangents<T>), dim3(grid_for(ctx, d.g.nmesh)), dim3(RED_THREADS),
                         0, ctx.stream, d.F.get(), d.G.get(), d.g.nmesh, d.nt, da.get());
      TRVG_LAUNCH_CHECK();
    }
    {
      std::unique_ptr<MeshScope> scope;
      if (d.coarse) scope = std::make_unique<MeshScope>(ctx, d.g);
      slab_fft<T>(ctx, d.F.get(), d.nt + 1);
    }
    ProfScope ps(ctx, KC_MISC, 3. * double(d.g.nmesh) * sizeof(c2<T>));
    hipLaunchKernelGGL((k_adj_acc<T>), dim3(grid_for(ctx, d.g.nmesh)), dim3(RED_THREADS), 0,
                       ctx.stream, acc.get(), d.F.get(), d.nt, g, d.g, ctx.tab, dedge.get(),
                       nb, dslot.get(), 1. / g.vol);
    TRVG_LAUNCH_CHECK();
    ctx.keep_until_flush(std::move(da));
    ctx.keep_until_flush(std::move(dslot));
  }
  // The products F_b^2 reach twice the highest bin edge.
  Prune pr{};
  if (all_coarse) pr = make_prune(g, 2. * kb.bin_edges[nb]);
  fft3d<T>(ctx, acc.get(), LoadSame<T>{acc.get()}, +1, -1., &pr);
  hipLaunchKernelGGL((k_real_part<T>), dim3(grid), dim3(RED_THREADS), 0,
                     ctx.stream, grad_mesh, acc.get(), nm, g.vol_cell);
  TRVG_LAUNCH_CHECK();
  ctx.flush();
}

template <typename T, int ORDER>
static void diff_assign_order(Context& ctx, T* mesh, const double* pos,
                              const double* w, long long n, bool accumulate) {
  const long long nm = ctx.g.nmesh;
  if (!accumulate) {
    hipLaunchKernelGGL((k_zero_real<T>), dim3(grid_for(ctx, nm)), dim3(RED_THREADS),
                       0, ctx.stream, mesh, nm);
    TRVG_LAUNCH_CHECK();
  }
  if (n > 0) {
    ProfScope ps(ctx, KC_ASSIGN, double(n) * 32. + double(nm) * sizeof(T));
    hipLaunchKernelGGL((k_assign_real<T, ORDER>), dim3(grid_for(ctx, n, 16)),
                       dim3(256), 0, ctx.stream, mesh, pos, w, n, ctx.g);
    TRVG_LAUNCH_CHECK();
  }
  TRVG_HIP(hipStreamSynchronize(ctx.stream));
}

template <typename T>
void diff_assign(Context& ctx, T* mesh, const double* pos, const double* w,
                 long long n, bool accumulate) {
  switch (ctx.p.assignment_order) {
    case 1: diff_assign_order<T, 1>(ctx, mesh, pos, w, n, accumulate); break;
    case 2: diff_assign_order<T, 2>(ctx, mesh, pos, w, n, accumulate); break;
    case 3: diff_assign_order<T, 3>(ctx, mesh, pos, w, n, accumulate); break;
    default: diff_assign_order<T, 4>(ctx, mesh, pos, w, n, accumulate); break;
  }
}

template <typename T, int ORDER>
static void diff_assign_adjoint_order(Context& ctx, const T* gmesh,
                                      const double* pos, const double* w,
                                      long long n, double* gpos, double* gw) {
  if (n > 0) {
    ProfScope ps(ctx, KC_ASSIGN, double(n) * (32. + 32.));
    hipLaunchKernelGGL((k_assign_real_adjoint<T, ORDER>), dim3(grid_for(ctx, n, 16)),
                       dim3(256), 0, ctx.stream, gmesh, pos, w, n, ctx.g, gpos, gw);
    TRVG_LAUNCH_CHECK();
  }
  TRVG_HIP(hipStreamSynchronize(ctx.stream));
}

template <typename T>
void diff_assign_adjoint(Context& ctx, const T* gmesh, const double* pos,
                         const double* w, long long n, double* gpos, double* gw) {
  switch (ctx.p.assignment_order) {
    case 1: diff_assign_adjoint_order<T, 1>(ctx, gmesh, pos, w, n, gpos, gw); break;
    case 2: diff_assign_adjoint_order<T, 2>(ctx, gmesh, pos, w, n, gpos, gw); break;
    case 3: diff_assign_adjoint_order<T, 3>(ctx, gmesh, pos, w, n, gpos, gw); break;
    default: diff_assign_adjoint_order<T, 4>(ctx, gmesh, pos, w, n, gpos, gw); break;
  }
}

template std::vector<double> diff_bispec_forward<double>(
    Context&, const trvg_binning&, double, const double*, std::vector<int>&);
template std::vector<double> diff_bispec_forward<float>(
    Context&, const trvg_binning&, double, const float*, std::vector<int>&);
template void diff_bispec_backward<double>(Context&, const trvg_binning&, double,
                                           const double*, const double*, double*);
template void diff_bispec_backward<float>(Context&, const trvg_binning&, double,
                                          const float*, const double*, float*);
template void diff_assign<double>(Context&, double*, const double*, const double*,
                                  long long, bool);
template void diff_assign<float>(Context&, float*, const double*, const double*,
                                 long long, bool);
template void diff_assign_adjoint<double>(Context&, const double*, const double*,
                                          const double*, long long, double*, double*);
template void diff_assign_adjoint<float>(Context&, const float*, const double*,
                                         const double*, long long, double*, double*);

}  // namespace trvg

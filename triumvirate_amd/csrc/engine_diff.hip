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
#include <algorithm>
#include <cmath>
#include <vector>

#include "diff_kernels.hpp"
#include "engine.hpp"

namespace trvg {

namespace {

// Bytes of one slab of shell fields, and of buffers waiting for the stream
// before the call waits for it.  Meshes up to 256^3 batch a group's bins whole
// or in a few parts, where launches count; larger ones take them two by two,
// so that a call needs three complex meshes (four and a real one with
// gradients) however many bins there are: 1024^3 FP64 52 and 77 GB.
constexpr size_t SLAB_BYTES = size_t(1) << 30;
constexpr size_t HELD_BYTES = size_t(2) << 30;

// The bins that share one mesh (every bin pairs with itself only).
struct DiffGroup {
  std::vector<int> bins;
  Geom g;
  bool coarse;
};

std::vector<DiffGroup> diff_groups(const Geom& g, const trvg_binning& kb,
                                   const std::vector<int>& bins, size_t cell) {
  std::vector<DiffGroup> out;
  for (const MeshGroup& gr : plan_mesh_groups(g, kb, bins, bins, true, cell)) {
    DiffGroup d;
    for (int q : gr.pairs) d.bins.push_back(bins[q]);   // a bin pairs with itself
    const Geom c = mesh_of(g, gr.n);
    // A smaller mesh has its own D(k): past 0.7 of the cells it takes more
    // memory than the full one saves.
    d.coarse = gr.coarse && (size_t(g.nmesh) * cell <= HELD_BYTES ||
                             double(c.nmesh) <= 0.7 * double(g.nmesh));
    d.g = d.coarse ? c : g;
    out.push_back(std::move(d));
  }
  return out;
}

// G(x) and the shell fields of one group: two real fields per complex mesh (bin
// q of a batch is component q % 2 of mesh q / 2), in batches of a slab.  D: the
// spectrum on the full mesh.
template <typename T>
class DiffFields {
 public:
  // spare: one more mesh in the slab if the group fits it whole.
  DiffFields(Context& ctx, const trvg_binning& kb, const DiffGroup& d, const c2<T>* D,
             bool spare)
      : ctx_(ctx), kb_(kb), d_(d), src_(D) {
    if (d.coarse) {
      cut_.reset(d.g.nmesh);
      truncate_modes<T>(ctx, D, d.g, cut_.get());
      src_ = cut_.get();
    }
    const size_t mesh = size_t(d.g.nmesh) * sizeof(c2<T>);
    const size_t nt = (d.bins.size() + 1) / 2, fit = std::max<size_t>(1, SLAB_BYTES / mesh);
    whole_ = nt + (spare ? 1 : 0) <= fit;
    per_ = int(whole_ ? nt : std::min(nt, fit));
    G_.reset(d.g.nmesh);
    F_.reset((per_ + (whole_ && spare ? 1 : 0)) * size_t(d.g.nmesh));
    auto scope = enter();
    fft3d<T>(ctx, G_.get(), LoadDeconv<T, T>{src_, ctx.tab, 1. / d.g.vol}, +1);
  }
  // Runs what follows on the group's mesh.
  std::unique_ptr<MeshScope> enter() {
    return d_.coarse ? std::make_unique<MeshScope>(ctx_, d_.g) : nullptr;
  }
  // fn(bins of a batch, meshes of it) with the batch's shell fields in F().
  template <class F>
  void batches(const std::vector<int>& nmodes, F fn) {
    for (size_t q = 0; q < d_.bins.size(); q += 2 * per_) {
      const std::vector<int> b(d_.bins.begin() + q,
                               d_.bins.begin() + std::min(q + 2 * per_, d_.bins.size()));
      {
        auto scope = enter();
        shell_slab_ifft<T, T>(ctx_, F_.get(), src_, kb_, b, nmodes, 0, 0, true);
      }
      fn(b, (int(b.size()) + 1) / 2);
    }
  }
  bool whole() const { return whole_; }
  c2<T>* F() { return F_.get(); }
  const c2<T>* G() const { return G_.get(); }
  // Leaves the buffers to the next flush, which comes now if much is held.
  void release(size_t& held) {
    held += (cut_.size() + G_.size() + F_.size()) * sizeof(c2<T>);
    ctx_.keep_until_flush(std::move(cut_));
    ctx_.keep_until_flush(std::move(G_));
    ctx_.keep_until_flush(std::move(F_));
    if (held > HELD_BYTES) {
      ctx_.flush();
      held = 0;
    }
  }

 private:
  Context& ctx_;
  const trvg_binning& kb_;
  const DiffGroup& d_;
  const c2<T>* src_;
  DevArray<c2<T>> cut_, G_, F_;
  bool whole_ = false;
  int per_ = 1;
};

// D(k) of the mesh.
template <typename T>
DevArray<c2<T>> diff_spectrum(Context& ctx, const T* mesh) {
  DevArray<c2<T>> D(ctx.g.nmesh);
  fft3d<T>(ctx, D.get(), LoadReal<T>{mesh, T(ctx.g.vol_cell)}, -1,
           double(ctx.g.nmesh) * sizeof(T));
  return D;
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
  DevArray<c2<T>> D = diff_spectrum<T>(ctx, mesh);
  std::vector<double> out(kb.num_bins);
  size_t held = 0;
  for (const DiffGroup& d : diff_groups(ctx.g, kb, bins, sizeof(c2<T>))) {
    DiffFields<T> f(ctx, kb, d, D.get(), false);
    f.batches(ss.nmodes, [&](const std::vector<int>& b, int nt) {
      const int nv = 2 * nt;
      const unsigned grid = grid_for(ctx, d.g.nmesh, 4);
      DevArray<double> part((size_t)grid * nv), sums(nv);   // [grid][nv]
      {
        ProfScope ps(ctx, KC_PAIR_REDUCE, double(nt + 1) * double(d.g.nmesh) * sizeof(c2<T>));
        hipLaunchKernelGGL((k_f2g_packed<T>), dim3(grid, unsigned(nt)), dim3(RED_THREADS), 0,
                           ctx.stream, f.F(), f.G(), d.g.nmesh, part.get());
        TRVG_LAUNCH_CHECK();
      }
      reduce_cols(ctx, part.get(), int(grid), nv, sums.get());
      const double* h = ctx.download(sums.get(), nv);
      ctx.keep_until_flush(std::move(part));
      ctx.keep_until_flush(std::move(sums));
      ctx.defer([h, b, vc = d.g.vol_cell, norm, &out, &ss] {
        for (size_t i = 0; i < b.size(); i++) {
          const double n = double(ss.nmodes[b[i]]);
          out[b[i]] = norm * vc * h[i] / (n * n);   // NaN for an empty bin
        }
      });
    });
    f.release(held);
  }
  ctx.flush();
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
  DevArray<c2<T>> D = diff_spectrum<T>(ctx, mesh);
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
  size_t held = 0;
  for (const DiffGroup& d : diff_groups(g, kb, bins, sizeof(c2<T>))) {
    all_coarse = all_coarse && d.coarse;
    // The cotangent of G is the slab's last mesh and is transformed with the
    // shells, or, over several batches, a real mesh transformed after them.
    DiffFields<T> f(ctx, kb, d, D.get(), true);
    DevArray<T> gG;
    if (!f.whole()) {
      gG.reset(d.g.nmesh);
      hipLaunchKernelGGL((k_zero_real<T>), dim3(grid_for(ctx, d.g.nmesh)), dim3(RED_THREADS), 0,
                         ctx.stream, gG.get(), d.g.nmesh);
      TRVG_LAUNCH_CHECK();
    }
    DevArray<int> dslot(nb);
    // acc += the spectra of the nt shell cotangents in F (slots `slot`) and
    // of that of G at gk (null: not yet).
    auto accumulate = [&](const std::vector<int>& slot, const c2<T>* gk) {
      ctx.upload(dslot.get(), slot.data(), nb);
      ProfScope ps(ctx, KC_MISC, 3. * double(d.g.nmesh) * sizeof(c2<T>));
      hipLaunchKernelGGL((k_adj_acc<T>), dim3(grid_for(ctx, d.g.nmesh)), dim3(RED_THREADS), 0,
                         ctx.stream, acc.get(), f.F(), gk, g, d.g, ctx.tab, dedge.get(), nb,
                         dslot.get(), 1. / g.vol);
      TRVG_LAUNCH_CHECK();
    };
    f.batches(ss.nmodes, [&](const std::vector<int>& b, int nt) {
      std::vector<double> a(2 * nt, 0.);
      std::vector<int> slot(nb, -1);
      for (size_t i = 0; i < b.size(); i++) {
        const double n = double(ss.nmodes[b[i]]);
        a[i] = grad_bk[b[i]] * norm * d.g.vol_cell / (n * n);
        slot[b[i]] = int(i);
      }
      DevArray<double> da(a.size());
      ctx.upload(da.get(), a.data(), a.size());
      c2<T>* gk = f.whole() ? f.F() + (long long)nt * d.g.nmesh : nullptr;
      {
        ProfScope ps(ctx, KC_MISC, (2. * nt + 2.) * double(d.g.nmesh) * sizeof(c2<T>));
        hipLaunchKernelGGL((k_cotangents<T>), dim3(grid_for(ctx, d.g.nmesh)), dim3(RED_THREADS),
                           0, ctx.stream, f.F(), f.G(), d.g.nmesh, nt, da.get(), gk, gG.get());
        TRVG_LAUNCH_CHECK();
      }
      {
        auto scope = f.enter();
        slab_fft<T>(ctx, f.F(), nt + (gk ? 1 : 0));
      }
      accumulate(slot, gk);
      ctx.keep_until_flush(std::move(da));
    });
    if (!f.whole()) {
      {
        auto scope = f.enter();
        fft3d<T>(ctx, f.F(), LoadReal<T>{gG.get(), T(1)}, -1, double(d.g.nmesh) * sizeof(T));
      }
      accumulate(std::vector<int>(nb, -1), f.F());
    }
    ctx.keep_until_flush(std::move(dslot));
    ctx.keep_until_flush(std::move(gG));
    f.release(held);
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

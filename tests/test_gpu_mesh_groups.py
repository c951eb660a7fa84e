"""Pair sums of band-limited bins on smaller meshes: the sums over the mesh
chosen for a group of pairs equal those over the full mesh, against the
oracle (which always sums over the full mesh).

The top edge h (in fundamental modes) of the bins sets the mesh: with
K = 2 h the 64^3 mesh is left for 32^3 up to K = 15, for 36^3 at K = 16 and
17, and kept from K = 30; at K >= 32 triples with k1 + k2 + k3 = +-n enter.
Diagonal, off-diagonal and row forms may split their pairs over several
meshes.

Tolerances: FP64 1e-10 of max |B| of the multipole; FP32 against FP64 1e-5;
gradients 1e-10 of the largest |gradient| (FP64 transforms of <= 64^3 cells
round at ~1e-15; 1e-10 is the bound of every engine-oracle comparison).
"""

import numpy as np
import pytest

import conftest as cf
import parity as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def backends():
    import oracle
    from triumvirate_amd import _lib
    from triumvirate_amd.threept import CLibBackend
    return CLibBackend(_lib.load()), oracle.backend(schedule=1)


def _run(be, deg, form, idx, geo, ng, top, precision='fp64'):
    from triumvirate_amd import threept as T
    from triumvirate_amd.dataobjs import Binning
    cell = 12.5
    box = [cell * n for n in ng]
    kf = 2 * np.pi / min(box)
    ps = cf.make_test_paramset(assignment='tsc', ngrid=dict(zip('xyz', ng)),
                               boxsize=dict(zip('xyz', box)))
    b = Binning('fourier', 'lin', bin_min=1.1 * kf, bin_max=(top + 0.01) * kf,
                num_bins=4)
    kw = dict(paramset=ps, degrees=deg, binning=b, form=form, idx_bin=idx,
              precision=precision)
    if geo == 'gpp':
        d = P.uniform_box_catalogue(4000, min(box), seed=5, weights=False)
        return T._compute_3pt_stats_sim_like(be, 'bispec', d, **kw)
    d, r = P.survey_pair(2000, 8000, 0.9 * min(box), seed=9, weights=True)
    return T._compute_3pt_stats_survey_like(be, 'bispec', d, r, **kw)


CASES = [
    # (degrees, form, idx, geometry, mesh, top edge in modes)
    ((0, 0, 0), 'full', None, 'gpp', (64, 64, 64), 7),
    ((0, 0, 0), 'full', None, 'gpp', (64, 64, 64), 8),
    ((0, 0, 0), 'diag', None, 'gpp', (64, 64, 64), 14),
    ((0, 0, 0), 'diag', None, 'gpp', (64, 64, 64), 15),
    ((0, 0, 0), 'diag', None, 'gpp', (64, 64, 64), 16),
    ((2, 0, 2), 'full', None, 'lpp', (64, 64, 64), 7),
    ((2, 0, 2), 'diag', None, 'lpp', (64, 64, 64), 20),
    ((1, 1, 0), 'row', 1, 'lpp', (64, 64, 64), 9),
    ((2, 0, 2), 'off-diag', 1, 'gpp', (64, 64, 64), 9),
    ((0, 2, 2), 'row', 0, 'lpp', (40, 64, 96), 6),
    ((0, 0, 0), 'diag', None, 'gpp', (96, 36, 64), 9),
]


@pytest.mark.parametrize('case', CASES, ids=['-'.join(map(str, c)) for c in CASES])
def test_mesh_groups_match_oracle(backends, case):
    print(f"mesh groups {case}", flush=True)
    a = _run(backends[0], *case)
    P.compare_results(a, _run(backends[1], *case), 'bispec', rtol=1e-10)
    f = _run(backends[0], *case, precision='fp32')
    for key in ('bk_raw', 'bk_shot'):
        err = np.max(np.abs(f[key] - a[key])) / np.max(np.abs(a[key]))
        assert err < 1e-5, (key, err)


@pytest.mark.parametrize('ng,top', [((64, 64, 64), 7), ((64, 64, 64), 15),
                                    ((64, 64, 64), 16), ((64, 64, 64), 30),
                                    ((64, 32, 128), 9)])
def test_gradients_on_smaller_meshes(ng, top):
    """Values and mesh gradients of the differentiable B_000 against the
    same sums written in torch over the full mesh."""
    import torch
    from triumvirate_amd.autodiff import DifferentiableBispectrum
    from triumvirate_amd.dataobjs import Binning
    print(f"gradients on smaller meshes {ng} {top}", flush=True)
    box = [12.5 * n for n in ng]
    kf = 2 * np.pi / min(box)
    b = Binning('fourier', 'lin', bin_min=1.1 * kf, bin_max=(top + 0.01) * kf,
                num_bins=5)
    g = torch.Generator().manual_seed(3)
    mesh = torch.randn(ng, generator=g, dtype=torch.float64)
    c = torch.randn(5, generator=g, dtype=torch.float64)
    k = [2 * np.pi * torch.fft.fftfreq(n, 1. / n, dtype=torch.float64) / L
         for n, L in zip(ng, box)]
    k = [k[0][:, None, None], k[1][None, :, None], k[2][None, None, :]]
    W = 1.
    for ka, L, n in zip(k, box, ng):
        u = ka * L / n / 2.
        W = W * torch.where(u == 0., torch.ones_like(u), u.sin() / u) ** 2
    km = (k[0] * k[0] + k[1] * k[1] + k[2] * k[2]).sqrt()
    vol, nm = np.prod(box), np.prod(ng)
    ref = mesh.clone().requires_grad_(True)
    D = torch.fft.fftn(ref) * (vol / nm) / W
    G = torch.fft.ifftn(D, norm='forward').real / vol
    want = []
    for i in range(5):
        sh = ((km >= b.bin_edges[i]) & (km < b.bin_edges[i + 1])).double()
        F = torch.fft.ifftn(D * sh, norm='forward').real
        want.append((vol / nm) * (F * F * G).sum() / sh.sum() ** 2)
    want = torch.stack(want)
    (want * c).sum().backward()
    x = mesh.cuda().requires_grad_(True)
    got = DifferentiableBispectrum(box, ng, b, 'cic', 'fp64').from_mesh(x)
    (got * c.cuda()).sum().backward()
    ref_g, want = ref.grad.numpy(), want.detach().numpy()
    assert np.max(np.abs(got.detach().cpu().numpy() - want)) < 1e-10 * np.max(np.abs(want))
    assert np.max(np.abs(x.grad.cpu().numpy() - ref_g)) < 1e-10 * np.max(np.abs(ref_g))


@pytest.mark.parametrize('prec', ['fp64', 'fp32'])
def test_bins_without_a_cotangent_are_left_out(prec):
    """A gradient of zero cotangents is zero, also of a mesh with a NaN, and a
    one-hot cotangent gives the gradient of a call on that bin alone."""
    import torch
    from triumvirate_amd.autodiff import DifferentiableBispectrum
    from triumvirate_amd.dataobjs import Binning
    print(f"bins without a cotangent {prec}", flush=True)
    ng, box = [32] * 3, [400.] * 3
    kf = 2 * np.pi / 400.
    b = Binning('fourier', 'lin', bin_min=1.1 * kf, bin_max=15.1 * kf, num_bins=5)
    one = Binning('fourier', 'lin', bin_min=b.bin_edges[3], bin_max=b.bin_edges[4],
                  num_bins=1)
    x = torch.randn(ng, generator=torch.Generator().manual_seed(4),
                    dtype=torch.float64).cuda()

    def grad(binning, c, x):
        x = x.to(torch.float32 if prec == 'fp32' else torch.float64)
        x = x.clone().requires_grad_(True)
        bk = DifferentiableBispectrum(box, ng, binning, 'cic', prec).from_mesh(x)
        bk.backward(torch.tensor(c, dtype=torch.float64).to(bk.device))
        return x.grad

    bad = x.clone()
    bad[1, 2, 3] = float('nan')
    assert not grad(b, [0.] * 5, bad).any()
    got, want = grad(b, [0., 0., 0., 2., 0.], x), grad(one, [2.], x)
    tol = 1e-12 if prec == 'fp64' else 1e-6   # pruning: rounding of empty modes
    assert (got - want).abs().max() < tol * want.abs().max()


def test_gradient_memory_does_not_grow_with_bins():
    """42 bins up to the Nyquist wavenumber of 256^3 FP64 (256 MiB a complex
    mesh): values and gradient add up from calls on 6 bins each, which take
    their shells in one slab, and the engine holds less than 3 GiB (all shells at
    once: 21 meshes, 5.3 GiB, beside the spectrum, G and the gradient)."""
    import torch
    from triumvirate_amd import _lib
    from triumvirate_amd.autodiff import DifferentiableBispectrum
    from triumvirate_amd.dataobjs import Binning
    print("gradient memory", flush=True)
    lib, ng, box = _lib.load(), [256] * 3, [1000.] * 3
    kf = 2 * np.pi / 1000.
    edges = np.linspace(1.1 * kf, 127.1 * kf, 43)
    g = torch.Generator(device='cuda').manual_seed(4)
    mesh = torch.randn(ng, generator=g, dtype=torch.float64, device='cuda')
    c = torch.randn(42, generator=g, dtype=torch.float64, device='cuda')

    def call(lo, hi):
        b = Binning('fourier', 'lin')
        b.set_custom_bins(edges[lo:hi + 1])
        x = mesh.clone().requires_grad_(True)
        bk = DifferentiableBispectrum(box, ng, b, 'cic', 'fp64').from_mesh(x)
        bk.backward(c[lo:hi])
        return bk.detach(), x.grad

    call(0, 1)                                   # what stays for the process
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    assert lib.trvg_release_workspace() == 0
    free, own = torch.cuda.mem_get_info()[0], torch.cuda.memory_reserved()
    bk, grad = call(0, 42)
    torch.cuda.synchronize()
    held = free - torch.cuda.mem_get_info()[0] - (torch.cuda.memory_reserved() - own)
    print(f"  {held / 2 ** 30:.2f} GiB", flush=True)
    assert held < 3 << 30
    want_g, want = torch.zeros_like(grad), []
    for lo in range(0, 42, 6):
        v, d = call(lo, lo + 6)
        want.append(v)
        want_g += d
    want = torch.cat(want)
    assert (bk - want).abs().max() < 1e-12 * want.abs().max()
    assert (grad - want_g).abs().max() < 1e-12 * want_g.abs().max()
    assert lib.trvg_release_workspace() == 0


def test_mixed_forms_share_bounded_slabs():
    """Multipoles of several forms in one call, where diagonal and row pairs go
    to smaller meshes: each equals its own call, in both precisions, and the
    slabs kept stay those of the full mesh, three of 20 complex fields
    (128^3 FP64: 1.9 GiB; the (2, m) of all terms together are four and a
    half), whatever the number of meshes."""
    import torch
    from triumvirate_amd import _lib
    from triumvirate_amd.dataobjs import Binning
    from triumvirate_amd.threept import (compute_bispec_in_gpp_box,
                                         compute_bispec_multipoles)
    print("mixed forms", flush=True)
    lib = _lib.load()
    kf = 2 * np.pi / 1000.
    b = Binning('fourier', 'lin', bin_min=1.1 * kf, bin_max=60. * kf, num_bins=20)
    ps = cf.make_test_paramset(assignment='cic', ngrid=dict.fromkeys('xyz', 128),
                               boxsize=dict.fromkeys('xyz', 1000.))
    mps = [((2, 2, 0), 'full'), ((0, 0, 0), 'diag'), ((2, 0, 2), 'row', 3),
           ((1, 1, 0), 'off-diag', 2)]

    def data():
        return P.uniform_box_catalogue(20000, 1000., seed=5, weights=False)

    for prec, tol in (('fp64', 1e-12), ('fp32', 1e-5)):
        torch.cuda.synchronize()
        assert lib.trvg_release_workspace() == 0
        free = torch.cuda.mem_get_info()[0]
        got = compute_bispec_multipoles(data(), multipoles=mps[:2], binning=b,
                                        paramset=ps, precision=prec)
        held = (free - torch.cuda.mem_get_info()[0]) / 2 ** 30
        print(f"  {prec} {held:.2f} GiB", flush=True)
        if prec == 'fp64':
            assert held < 2.8
        got = compute_bispec_multipoles(data(), multipoles=mps, binning=b,
                                        paramset=ps, precision=prec)
        for mp, res in zip(mps, got):
            one = compute_bispec_in_gpp_box(
                data(), degrees=mp[0], form=mp[1], idx_bin=mp[2] if len(mp) > 2 else None,
                binning=b, paramset=ps, precision=prec)
            for key in ('bk_raw', 'bk_shot'):
                err = np.max(np.abs(res[key] - one[key])) / np.max(np.abs(one[key]))
                assert err < tol, (mp, key, err)
    assert lib.trvg_release_workspace() == 0

"""FP32 pair sums on the matrix cores (16 x 16 pairs per tile, at most two
tiles a side per launch) against the FP64 engine, whose pair sums run on the
vector units.

Numbers of bins at the tile edges (1, 15, 16, 17, 32, 33), every kind of
sides (real with real, complex with real in both orders, complex with
complex; real, imaginary and full complex sums) and meshes whose cell count
is and is not a multiple of the kernel's 128-cell chunk.  Tolerance, of max
|zeta|: the fields of a catalogue of noise are rounded at about 4e-7 by their
FP32 transforms, and their sums cancel to about 1 / sqrt(cells) of the sum of
magnitudes, so 4e-7 sqrt(cells) (2.6e-5 at 16^3, 2.1e-5 at 14^3); a pair or a
cell summed wrongly shows at 1 / cells or more.
"""

import numpy as np
import pytest

import conftest as cf
import parity as P

pytestmark = pytest.mark.gpu

# degrees: sides of its terms
DEGREES = [
    (0, 0, 0),   # real x real, one slab
    (2, 0, 2),   # complex x real, real parts; real x real, two slabs
    (1, 1, 0),   # complex x complex, real parts and full sums
    (1, 0, 1),   # complex x real, imaginary parts and full sums
    (2, 1, 1),   # real x complex, complex x complex, imaginary parts
]


@pytest.mark.parametrize('degrees', DEGREES, ids=lambda d: ''.join(map(str, d)))
@pytest.mark.parametrize('nb,ng', [(1, 16), (15, 14), (16, 16), (17, 14),
                                   (32, 16), (33, 14)])
def test_fp32_pair_sums_match_fp64(degrees, nb, ng):
    from triumvirate_amd import _lib
    from triumvirate_amd import threept as T
    from triumvirate_amd.dataobjs import Binning
    print(f"pair sums {degrees} bins {nb} mesh {ng}", flush=True)
    be = T.CLibBackend(_lib.load())
    ps = cf.make_test_paramset(assignment='cic', ngrid=dict.fromkeys('xyz', ng),
                               boxsize=dict.fromkeys('xyz', 400.))
    b = Binning('config', 'lin', bin_min=30., bin_max=180., num_bins=nb)
    out = []
    for precision in ('fp32', 'fp64'):
        d, r = P.survey_pair(1500, 4000, 360., seed=9, weights=True)
        out.append(T._compute_3pt_stats_survey_like(
            be, '3pcf', d, r, paramset=ps, degrees=degrees, binning=b, form='full',
            precision=precision))
    scale = np.max(np.abs(out[1]['zeta_raw']))
    err = np.max(np.abs(out[0]['zeta_raw'] - out[1]['zeta_raw'])) / scale
    print(f"  {err:.2e}", flush=True)
    assert err < 4e-7 * ng ** 1.5


@pytest.mark.parametrize('precision,eps', [('fp64', 4e-15), ('fp32', 4e-7)])
@pytest.mark.parametrize('degrees', DEGREES, ids=lambda d: ''.join(map(str, d)))
@pytest.mark.parametrize('form,idx', [('diag', 0), ('off-diag', 1), ('row', 2)])
@pytest.mark.parametrize('nb,ng', [(4, 14), (9, 16), (17, 18)])
def test_pair_lists_match_full_tables(degrees, precision, eps, form, idx, nb, ng):
    """Lists of about one pair per field are streamed; the same pairs of the
    full table come from the tiled kernels.  Batches of eight pairs: lists of
    3 to 17, meshes with a remainder.  The fields are the same, the sums cancel
    as above: eps sqrt(cells) of max |zeta| (eps ten roundings in FP64)."""
    from triumvirate_amd import _lib
    from triumvirate_amd import threept as T
    from triumvirate_amd.dataobjs import Binning
    print(f"pair lists {degrees} {precision} {form} bins {nb} mesh {ng}", flush=True)
    be = T.CLibBackend(_lib.load())
    ps = cf.make_test_paramset(assignment='cic', ngrid=dict.fromkeys('xyz', ng),
                               boxsize=dict.fromkeys('xyz', 400.))
    b = Binning('config', 'lin', bin_min=30., bin_max=180., num_bins=nb)
    out = []
    for f in (form, 'full'):
        d, r = P.survey_pair(1500, 4000, 360., seed=9, weights=True)
        out.append(T._compute_3pt_stats_survey_like(
            be, '3pcf', d, r, paramset=ps, degrees=degrees, binning=b, form=f,
            idx_bin=idx, precision=precision)['zeta_raw'])
    assert np.isfinite(out[0]).all() and np.isfinite(out[1]).all()
    if out[1].size == nb * nb:
        full, known = out[1].reshape(nb, nb), np.full((nb, nb), True)
    else:                      # equal degrees: only the upper triangle
        known = np.triu(np.full((nb, nb), True))
        full = np.zeros((nb, nb), out[1].dtype)
        full[known] = out[1]
        if degrees == (0, 0, 0):           # symmetric in its two sides
            full, known = full + np.triu(full, 1).T, np.full((nb, nb), True)
    cut = {'diag': np.diag, 'off-diag': lambda a: np.diag(a, idx),
           'row': lambda a: a[idx]}[form]
    want, known = cut(full), cut(known)
    assert out[0].shape == want.shape and known.sum() >= nb - 2
    err = np.max(np.abs(out[0] - want)[known]) / np.max(np.abs(full))
    print(f"  {err:.2e}", flush=True)
    assert err < eps * ng ** 1.5

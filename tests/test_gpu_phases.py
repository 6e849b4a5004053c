"""Queries on both sides of the lines where their phases, their sample pass and
their last tile's lists change: the rows of the contraction forms equal the
exact form's bit for bit."""
import numpy as np
import pytest

from mdsctk_amd import knn, synth

pytestmark = pytest.mark.gpu


def _rows(prec, ref, w, queries):
    with knn.KnnContext(0, prec) as ctx:
        ctx.set_reference(ref, w)
        return [ctx.query(x, k, flags) for x, k, flags in queries]


@pytest.mark.parametrize("prec", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("n_ref,natoms", [(127, 33), (1000, 40), (3001, 150), (5500, 65), (8200, 20)])
def test_nofit_and_fitted_rows_equal_the_exact_form(n_ref, natoms, prec):
    """One tile an item, several, an odd last pair; lists of 2 to 41 entries;
    one to sixteen blocks of 128 query frames."""
    x = synth.metastable_trajectory(n_ref + 2000, natoms, n_ref + natoms, n_centres=9)
    ref, fit = x[:n_ref], x[n_ref:]
    w = synth.masses(natoms, "random", 1)
    queries = [(fit[:m], k, f) for m in (33, 128, 129, 300, 2000) for k in (1, 4, 10, 40)
               for f in (knn.KNN_NOFIT, 0) if not (m == 2000 and n_ref > 5000 and f == 0)]
    for (d, i), (d_e, i_e) in zip(_rows(prec, ref, w, queries), _rows("exact", ref, w, queries)):
        np.testing.assert_array_equal(i, i_e)
        np.testing.assert_array_equal(d, d_e)


@pytest.mark.parametrize("flags", [0, knn.KNN_NOFIT])
@pytest.mark.parametrize("n,k", [(4096, 3), (4200, 120), (7000, 20), (17000, 8)])
def test_self_rows_with_a_band_pass_over_several_lists(n, k, flags):
    frames = synth.metastable_trajectory(n, 24, n, n_centres=15)
    d, i = _rows("bf16", frames, None, [(None, k, flags)])[0]
    d_e, i_e = _rows("exact", frames, None, [(frames[::7], k, flags)])[0]
    np.testing.assert_array_equal(i[::7], i_e)
    np.testing.assert_array_equal(d[::7], d_e)


@pytest.mark.parametrize("n_ref,natoms", [(16400, 256), (16400, 257), (32768, 300), (32767, 300)])
def test_short_fp32_rows_equal_the_exact_form(n_ref, natoms):
    """With a sample pass and without, by frame length, rows and references."""
    x = synth.metastable_trajectory(n_ref + 255, natoms, 5, n_centres=9)
    ref, fit = x[:n_ref], x[n_ref:]
    w = synth.masses(natoms, "random", 1)
    queries = [(fit[:m], k, 0) for m in (1, 31, 32, 255) for k in (1, 40)]
    for (d, i), (d_e, i_e) in zip(_rows("fp32", ref, w, queries), _rows("exact", ref, w, queries)):
        np.testing.assert_array_equal(i, i_e)
        np.testing.assert_array_equal(d, d_e)

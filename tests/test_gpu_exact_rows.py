"""Whole rows of exact scores at the edges of their kernel's tiling: 4 query
rows and 32 references per workgroup, atoms staged 256 at a time, 16 lanes a
pair.  Full rows (--sort false), the exact form and the re-scored candidate
lists must agree bit for bit on every pair, and with the FP64 oracle."""
import numpy as np
import pytest

import oracle
from mdsctk_amd import knn, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natoms", [1, 15, 16, 17, 255, 256, 257, 530])
@pytest.mark.parametrize("n_ref,n_fit", [(31, 1), (32, 4), (33, 5), (97, 3), (1030, 7)])
@pytest.mark.parametrize("flags", [0, knn.KNN_NOFIT])
def test_exact_rows_tiling(natoms, n_ref, n_fit, flags):
    x = synth.trajectory(n_ref + n_fit, natoms, 11 * natoms + n_ref)
    ref, fit = x[:n_ref], x[n_ref:]
    w = synth.masses(natoms, "random", 4)
    k = n_ref - 1
    with knn.KnnContext(0, "bf16") as ctx:
        ctx.set_reference(ref, w)
        full, ids = ctx.query(fit, 0, flags | knn.KNN_FULL_ROWS)
        d, i = ctx.query(fit, min(k, 100), flags)
    with knn.KnnContext(0, "exact") as ctx:
        ctx.set_reference(ref, w)
        d_e, i_e = ctx.query(fit, k, flags)
    np.testing.assert_array_equal(ids, np.broadcast_to(np.arange(n_ref), ids.shape))
    np.testing.assert_array_equal(np.take_along_axis(full, i_e.astype(np.int64), 1), d_e)
    np.testing.assert_array_equal(d, d_e[:, :d.shape[1]])
    np.testing.assert_array_equal(i, i_e[:, :i.shape[1]])
    # every row's sorted distances, rank 0 included, against the oracle's
    d_o, _ = oracle.knn_exact(ref, fit, w, k, nofit=bool(flags & knn.KNN_NOFIT))
    assert np.abs(d_e - d_o).max() < 1e-4

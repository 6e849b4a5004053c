"""Short queries: up to 32 frames take the contraction's one-fit-tile
workgroups, and fewer than 256 frames against 16384 or more resident frames
bound their thresholds with a sample pass.  Both sides of each limit must
return the rows of a longer query, and the FP64 oracle's."""
import numpy as np
import pytest

import oracle
from mdsctk_amd import knn, synth
from tests.parity import check_knn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("flags", [0, knn.KNN_NOFIT])
@pytest.mark.parametrize("n_ref,natoms,k", [(16383, 30, 9), (16384, 65, 50), (16500, 17, 300),
                                            (17001, 40, 800), (130, 200, 20)])
def test_short_queries(prec, flags, n_ref, natoms, k):
    x = synth.metastable_trajectory(n_ref + 300, natoms, 8, n_centres=9)
    if flags & knn.KNN_NOFIT:  # frames as given share no frame of reference
        x = (x - x.mean(axis=1, keepdims=True)).astype(np.float32)
    ref, fit = x[:n_ref], x[n_ref:]
    w = synth.masses(natoms, "random", 7)
    with knn.KnnContext(0, prec) as ctx:
        ctx.set_reference(ref, w)
        d0, i0 = ctx.query(fit, k, flags)
        for n in (1, 2, 31, 32, 33, 64, 65, 128, 129, 255, 256):
            d, i = ctx.query(fit[:n], k, flags)
            np.testing.assert_array_equal(i, i0[:n])
            np.testing.assert_array_equal(d, d0[:n])
        reqs = [ctx.wait(ctx.submit(fit[a:b], k, flags)) for a, b in ((0, 1), (1, 33), (33, 299))]
    got = np.concatenate([r.idx for r in reqs])
    np.testing.assert_array_equal(got, i0[:299])
    rows = np.arange(0, 300, 61)
    d_o, i_o = oracle.knn_exact(ref, fit[rows], w, k, nofit=bool(flags & knn.KNN_NOFIT))
    check_knn(ref, fit[rows], w, d0[rows], i0[rows], d_o, i_o, nofit=bool(flags & knn.KNN_NOFIT))

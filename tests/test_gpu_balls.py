"""The ball test before the tile filter, on both sides of the size up to which
it takes a self query's rows one by one: the symmetric query equals the list
path, which knows no test, bit for bit."""
import numpy as np
import pytest

from mdsctk_amd import knn, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,natoms,centres,k", [(65536, 6, 40, 10), (65537, 6, 40, 10),
                                                (4161, 52, 9, 70), (4097, 33, 65, 3)])
@pytest.mark.parametrize("prec", ["bf16", "fp32"])
def test_ball_test_equals_lists(n, natoms, centres, k, prec):
    x = synth.metastable_trajectory(n, natoms, 5, n_centres=centres)
    x[n // 2:n // 2 + 100] = x[7]  # balls of radius 0, and ties
    w = synth.masses(natoms, "random", 7)
    out = []
    for sym in (1, 0):
        with knn.KnnContext(0, prec) as ctx:
            ctx.set_option(knn.OPT_SELF_SYMMETRIC, sym)
            ctx.set_reference(x, w)
            out.append(ctx.query(None, k))
    np.testing.assert_array_equal(out[0][1], out[1][1])
    np.testing.assert_array_equal(out[0][0], out[1][0])

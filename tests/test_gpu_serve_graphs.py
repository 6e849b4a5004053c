"""Served batches of alternating sizes replay the executable graph of their
kind; none is built anew once every kind has been seen."""
import numpy as np
import pytest

from mdsctk_amd import knn, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flags", [0, knn.KNN_NOFIT])
def test_alternating_sizes_build_no_graphs(flags):
    n_ref, natoms, k = 22000, 300, 12
    x = synth.metastable_trajectory(n_ref + 2048, natoms, 3, n_centres=12)
    ref, fit = x[:n_ref], x[n_ref:]
    sizes = (1, 40, 300, 2048, 33, 256, 32, 257, 600, 1999)
    with knn.KnnContext(0, "bf16") as ctx:
        ctx.set_option(knn.OPT_SERVE_SLOTS, 1)
        ctx.set_reference(ref)
        for _ in range(5):  # the ordered copy
            want = ctx.query(fit, k, flags)
        built = []
        for _ in range(3):
            for m in sizes:
                r = ctx.wait(ctx.submit(fit[:m], k, flags))
                np.testing.assert_array_equal(r.idx, want[1][:m])
                np.testing.assert_array_equal(r.dist, want[0][:m])
            built.append(ctx.serve_stats()["graph_builds"])
        assert built[0] <= 8
        assert built[1] == built[0] and built[2] == built[0]

"""A memory budget set after a resident set was ordered for cross queries: the
ordered copy is given back, and the query's rows stay the same."""
import numpy as np
import pytest

from mdsctk_amd import knn, synth

pytestmark = pytest.mark.gpu


def test_budget_frees_the_ordered_copy():
    n_ref, natoms, k = 8200, 520, 12
    x = synth.metastable_trajectory(n_ref + 2100, natoms, 3, n_centres=12)
    ref, fit = x[:n_ref], x[n_ref:]
    w = synth.masses(natoms, "random", 2)
    with knn.KnnContext(0, "bf16") as ctx:
        ctx.set_reference(ref, w)
        d0, i0 = ctx.query(fit, k)
        plain = ctx.stats()["device_bytes"]
        for _ in range(4):
            d, i = ctx.query(fit, k)
        ordered = ctx.stats()["device_bytes"]
        assert ordered > plain
        ctx.set_option(knn.OPT_HBM_BUDGET, plain)
        d1, i1 = ctx.query(fit, k)
        assert ctx.stats()["device_bytes"] <= plain
        ctx.set_option(knn.OPT_HBM_BUDGET, 0)
        d2, i2 = ctx.query(fit, k)
    for a, b in ((d, i), (d1, i1), (d2, i2)):
        np.testing.assert_array_equal(b, i0)
        np.testing.assert_array_equal(a, d0)

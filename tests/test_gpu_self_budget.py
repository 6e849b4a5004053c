"""Self queries under memory budgets: the symmetric form is kept with fewer
candidate lists where they fit."""
import numpy as np
import pytest

from mdsctk_amd import knn, synth

pytestmark = pytest.mark.gpu

N, NATOMS, K = 6000, 64, 12


@pytest.fixture(scope="module")
def frames():
    return synth.metastable_trajectory(N, NATOMS, 9, n_centres=12)


def _query(frames, budget=0, mirror_cap=0):
    with knn.KnnContext(0, "bf16") as ctx:
        if mirror_cap:
            ctx.set_option(knn.OPT_MIRROR_CAP, mirror_cap)
        if budget:
            ctx.set_option(knn.OPT_HBM_BUDGET, budget)
        ctx.set_reference(frames)
        before = ctx.stats()["device_bytes"]
        rows = ctx.query(None, K)
        return rows, ctx.stats(), before


def test_symmetric_form_with_fewer_lists(frames):
    """Half the memory of the free query, and a third, hold the form with
    fewer phases (less only when not even four fit)."""
    want, st, base = _query(frames, mirror_cap=64)
    assert st["n_pairs_landmark"] > 0 and st["ref_splits"] == 16
    size = st["device_bytes"] - base
    for part, splits in ((1.01, 16), (0.75, 8), (0.55, 8), (0.45, 4), (0.34, 4)):
        rows, st, _ = _query(frames, int(base + part * size), 64)
        assert (st["n_pairs_landmark"] > 0, st["ref_splits"]) == (True, splits), part
        np.testing.assert_array_equal(rows[1], want[1])
        np.testing.assert_array_equal(rows[0], want[0])

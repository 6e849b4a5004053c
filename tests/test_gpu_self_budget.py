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


def test_rows_in_a_second_pass_fit_any_budget(frames):
    """Short mirrored lists overflow, and their rows go through the candidate
    lists once more: whatever the budget, also one that the first pass fills
    to the last bytes, the query returns its rows."""
    want, st, base = _query(frames, mirror_cap=8)
    assert st["n_relisted_rows"] > 1000
    size = st["device_bytes"] - base
    # the largest use of each number of phases, and just above and below
    for splits in (16, 8, 4):
        lo, hi = 0.02, 1.4
        for _ in range(22):
            mid = (lo + hi) / 2
            _, st, _ = _query(frames, int(base + mid * size), 8)
            if st["n_pairs_landmark"] and st["ref_splits"] >= splits:
                hi = mid
            else:
                lo = mid
        edge = int(base + hi * size)
        for budget in (edge - 70000, edge, edge + 1000, edge + 300000, edge + 4000000):
            rows, st, _ = _query(frames, budget, 8)
            np.testing.assert_array_equal(rows[1], want[1])
            np.testing.assert_array_equal(rows[0], want[0])

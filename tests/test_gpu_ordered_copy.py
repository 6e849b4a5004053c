"""When a context makes the ordered copy of its resident set, what it holds for
it, and when it gives it back.  Rows are the same with and without."""
import numpy as np
import pytest

from mdsctk_amd import knn, synth

pytestmark = pytest.mark.gpu

N_REF, NATOMS, K = 20000, 520, 12
COPY = 12 * N_REF * NATOMS  # bytes of the copy's operand alone


@pytest.fixture(scope="module")
def frames():
    x = synth.metastable_trajectory(N_REF + 2100, NATOMS, 3, n_centres=12)
    return x[:N_REF], x[N_REF:]


def _held(ctx):
    return ctx.stats()["device_bytes"]


def test_short_queries_do_not_make_the_copy(frames):
    """Queries below 256 frames never walk the copy, nor do those whose pairs
    are too few for it (800 frames here), however many there are."""
    ref, fit = frames
    for m in (255, 800):
        with knn.KnnContext(0, "bf16") as ctx:
            ctx.set_reference(ref)
            want = ctx.query(fit[:m], K)
            before = _held(ctx)
            for _ in range(9000 // m + 1):
                d, i = ctx.query(fit[:m], K)
            np.testing.assert_array_equal(i, want[1])
            assert _held(ctx) == before


def test_served_batches_of_growing_size_allocate_nothing(frames):
    """A slot's first batch against the ordered copy sizes its workspace for
    the largest one."""
    ref, fit = frames
    with knn.KnnContext(0, "bf16") as ctx:
        ctx.set_option(knn.OPT_SERVE_SLOTS, 1)
        ctx.set_reference(ref)
        want = ctx.query(fit, K)
        for _ in range(4):
            ctx.query(fit, K)
        ctx.wait(ctx.submit(fit[:1700], K))
        before = _held(ctx)
        for m in (900, 300, 1100, 2048, 1999):
            r = ctx.wait(ctx.submit(fit[:m], K))
            np.testing.assert_array_equal(r.idx, want[1][:m])
            np.testing.assert_array_equal(r.dist, want[0][:m])
            assert _held(ctx) == before


@pytest.mark.parametrize("busy", [False, True])
def test_budget_set_while_serving_gives_the_copy_back(frames, busy):
    """At once when no request is in flight, else with the next batch."""
    ref, fit = frames
    with knn.KnnContext(0, "bf16") as ctx:
        ctx.set_reference(ref)
        want = ctx.query(fit, K)
        plain = _held(ctx)
        for _ in range(4):
            ctx.query(fit, K)
        made = _held(ctx)
        assert made > plain + COPY
        reqs = [ctx.submit(fit, K) for _ in range(12)]
        if not busy:
            for r in reqs:
                ctx.wait(r)
        before = _held(ctx)
        ctx.set_option(knn.OPT_HBM_BUDGET, 64 << 30)
        if not busy:
            assert _held(ctx) < before - COPY
        for r in reqs + [ctx.submit(fit, K)]:
            ctx.wait(r)
            np.testing.assert_array_equal(r.idx, want[1])
            np.testing.assert_array_equal(r.dist, want[0])
        d, i = ctx.query(fit, K)
        np.testing.assert_array_equal(i, want[1])
        held = _held(ctx)
        # without the budget the copy comes back, and is what was missing
        ctx.set_option(knn.OPT_HBM_BUDGET, 0)
        for _ in range(5):
            d, i = ctx.query(fit, K)
        np.testing.assert_array_equal(i, want[1])
        np.testing.assert_array_equal(d, want[0])
        assert _held(ctx) > held + COPY


@pytest.mark.parametrize("prec", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("gen,n_ref,natoms,n_fit,k", [
    ("states", 16385, 260, 2500, 1), ("states", 16385, 260, 2300, 70), ("basin", 15000, 290, 2100, 12),
    ("loose", 10007, 420, 4097, 5), ("copies", 12000, 350, 3000, 30), ("states", 9000, 470, 17000, 9),
    ("states", 16385, 260, 4100, 70), ("basin", 15000, 290, 2700, 12), ("copies", 12000, 350, 3700, 30)])
def test_ordered_rows_equal_the_unordered_ones(gen, n_ref, natoms, n_fit, k, prec):
    """Blocks around one place and around many, unrelated frames (more places
    than a block's pass takes), a resident set of 40 frames' copies (equal
    keys), more query frames than the rank sort takes; on both sides of the
    length from which queries are ordered."""
    rng = np.random.default_rng(n_ref)
    n = n_ref + n_fit
    if gen == "states":
        x = synth.metastable_trajectory(n, natoms, 3, n_centres=50)
    elif gen == "basin":
        x = synth.trajectory(n, natoms, 4)
    elif gen == "loose":
        x = np.stack([synth.random_walk(natoms, rng) for _ in range(n)]).astype(np.float32)
    else:
        x = synth.metastable_trajectory(40, natoms, 3, n_centres=40)[rng.integers(0, 40, n)]
    ref, fit = x[:n_ref], x[n_ref:]
    w = synth.masses(natoms, "random", 2)
    with knn.KnnContext(0, prec) as ctx:
        ctx.set_option(knn.OPT_HBM_BUDGET, 200e9)  # no copy under a budget
        ctx.set_reference(ref, w)
        d0, i0 = ctx.query(fit, k)
        ctx.set_option(knn.OPT_HBM_BUDGET, 0)
        plain = _held(ctx)
        for _ in range(8192 // n_fit + 2):
            d, i = ctx.query(fit, k)
        assert _held(ctx) > plain + n_ref * natoms * (6 if prec == "fp32" else 12)
    np.testing.assert_array_equal(i, i0)
    np.testing.assert_array_equal(d, d0)

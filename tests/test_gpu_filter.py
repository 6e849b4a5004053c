"""The tile filter of fitted queries (filter_kernels.hip).  Self queries: from
4096 frames on, a proven bound decides which tiles of the block triangle are
contracted at all.  Outputs must equal the candidate-list path's bit for bit
and the FP64 oracle's, at the edges of the filter's layout: one and two
segments (384 atoms), one and two K-groups per stage (309), slots exactly
full and one over (52, 53, 116, 117), frames of 1 to 3 atoms, ragged frame
counts, and sets whose tiles all stay (a single basin with a wide k).  Cross
queries: once a context has seen enough query frames it orders the resident
set, and later queries (synchronous and served) walk the filtered tiles; they
must return what the first ones did."""
import numpy as np
import pytest

import oracle
from mdsctk_amd import knn, synth
from tests.parity import check_knn

pytestmark = pytest.mark.gpu


def _rows(frames, w, k, prec, sym, flags=0):
    with knn.KnnContext(0, prec) as ctx:
        ctx.set_option(knn.OPT_SELF_SYMMETRIC, sym)
        ctx.set_reference(frames, w)
        return ctx.query(None, k, flags)


def _check(frames, w, k, prec):
    d_s, i_s = _rows(frames, w, k, prec, 1)
    d_l, i_l = _rows(frames, w, k, prec, 0)
    np.testing.assert_array_equal(i_s, i_l)
    np.testing.assert_array_equal(d_s, d_l)
    rows = np.arange(0, len(frames), len(frames) // 5)
    d_o, i_o = oracle.knn_exact(frames, frames[rows], w, k)
    check_knn(frames, frames[rows], w, d_s[rows], i_s[rows], d_o, i_o)


@pytest.mark.parametrize("prec", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("natoms,n,k", [(52, 4096, 12), (53, 4097, 12), (116, 4225, 30),
                                        (117, 6000, 30), (308, 4160, 20), (309, 4159, 20),
                                        (383, 4321, 9), (384, 4321, 9), (700, 4500, 40)])
def test_filtered_self_query_on_states(natoms, n, k, prec):
    frames = synth.metastable_trajectory(n, natoms, natoms + n, n_centres=20)
    _check(frames, synth.masses(natoms, "random", 1), k, prec)


@pytest.mark.parametrize("natoms,n,k", [(1, 4200, 5), (2, 4200, 5), (3, 4200, 5), (30, 4200, 300),
                                        (400, 4300, 60)])
def test_filtered_self_query_on_one_basin(natoms, n, k):
    frames = synth.trajectory(n, natoms, 77 + natoms)
    _check(frames, synth.masses(natoms, "backbone"), k, "bf16")


@pytest.mark.parametrize("natoms", [60, 400])
def test_filtered_self_query_on_hard_frames(natoms):
    """Straight chains (two moments vanish), unrelated conformations (the
    deviations from the mean are as large as the frames), a run of equal
    frames, and coordinates far outside and far inside FP32's squares."""
    rng = np.random.default_rng(5)
    w = synth.masses(natoms, "wide", 3)
    _check(synth.extended_chain(4200, natoms, 4), w, 10, "bf16")
    loose = np.stack([synth.random_walk(natoms, rng) for _ in range(4200)]).astype(np.float32)
    _check(loose, w, 10, "bf16")
    loose[300:420] = loose[300]
    _check(loose, w, 10, "bf16")


@pytest.mark.parametrize("scale", [1e-8, 1e8])
def test_filtered_self_query_scales(scale):
    """The same set in other units gives the same neighbours."""
    frames = synth.metastable_trajectory(4200, 64, 9, n_centres=12)
    frames -= frames.mean(axis=1, keepdims=True)
    w = synth.masses(64, "uniform")
    d, i = _rows(frames, w, 8, "bf16", 1)
    power = np.float32(2.0 ** round(np.log2(scale)))
    d2, i2 = _rows(frames * power, w, 8, "bf16", 1)
    np.testing.assert_array_equal(i, i2)
    np.testing.assert_allclose(d2, d * float(power), rtol=1e-9)


@pytest.mark.parametrize("prec", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("gen,natoms,n_ref,n_fit,k", [("states", 470, 9001, 2100, 20),
                                                      ("basin", 513, 8192, 2085, 40),
                                                      ("loose", 600, 8300, 2300, 5)])
def test_ordered_cross_query(gen, natoms, n_ref, n_fit, k, prec):
    n = n_ref + n_fit
    if gen == "states":
        x = synth.metastable_trajectory(n, natoms, 3, n_centres=15)
    elif gen == "basin":
        x = synth.trajectory(n, natoms, 4)
    else:
        rng = np.random.default_rng(6)
        x = np.stack([synth.random_walk(natoms, rng) for _ in range(n)]).astype(np.float32)
    ref, fit = x[:n_ref], x[n_ref:]
    w = synth.masses(natoms, "random", 2)
    with knn.KnnContext(0, prec) as ctx:
        ctx.set_reference(ref, w)
        d0, i0 = ctx.query(fit, k)
        held = ctx.stats()["device_bytes"]
        for _ in range(4):
            d, i = ctx.query(fit, k)
            np.testing.assert_array_equal(i, i0)
            np.testing.assert_array_equal(d, d0)
        # the ordered copy of the resident set now exists
        assert ctx.stats()["device_bytes"] > held + 12 * n_ref * natoms
        for m in (255, 256, 257, 1000):  # either side of the smallest ordered query
            d, i = ctx.query(fit[:m], k)
            np.testing.assert_array_equal(i, i0[:m])
            np.testing.assert_array_equal(d, d0[:m])
        reqs = [ctx.submit(fit[a:b], k) for a, b in ((0, 1), (1, 900), (900, n_fit))]
        for r, (a, b) in zip(reqs, ((0, 1), (1, 900), (900, n_fit))):
            ctx.wait(r)
            np.testing.assert_array_equal(r.idx, i0[a:b])
            np.testing.assert_array_equal(r.dist, d0[a:b])
        d, i = ctx.query(fit, k, knn.KNN_KEEP_RANK0)
        np.testing.assert_array_equal(i[:, 1:], i0[:, :-1])
    rows = np.arange(0, n_fit, n_fit // 5)
    d_o, i_o = oracle.knn_exact(ref, fit[rows], w, k)
    check_knn(ref, fit[rows], w, d0[rows], i0[rows], d_o, i_o)


@pytest.mark.parametrize("power", [-18, -23, -24, -27, -31, -33, -34])
def test_filtered_self_query_of_tiny_frames(power):
    """G terms from 2e-9 down to 4e-19, on both sides of 1e-12, below which a
    frame's tiles are all kept: there the filter's FP32 squares reach the
    subnormal numbers.  No row may need a second pass either."""
    frames = synth.trajectory(4300, 64, 5)
    frames = (frames - frames.mean(axis=1, keepdims=True)) * np.float32(2.0 ** power)
    rows = []
    for sym in (1, 0):
        with knn.KnnContext(0, "bf16") as ctx:
            ctx.set_option(knn.OPT_SELF_SYMMETRIC, sym)
            ctx.set_reference(frames)
            rows.append(ctx.query(None, 8))
            st = ctx.stats()
            assert st["n_relisted_rows"] == 0 and st["n_fallback_rows"] == 0
    np.testing.assert_array_equal(rows[0][1], rows[1][1])
    np.testing.assert_array_equal(rows[0][0], rows[1][0])

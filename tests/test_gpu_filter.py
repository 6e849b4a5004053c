"""The tile filter of a fitted self query (filter_kernels.hip): from 4096
frames on, a proven bound decides which tiles of the block triangle are
contracted at all.  Outputs must equal the candidate-list path's bit for bit
and the FP64 oracle's, at the edges of the filter's layout: one and two
segments (384 atoms), one and two K-groups per stage (309), slots exactly
full and one over (52, 53, 116, 117), frames of 1 to 3 atoms, ragged frame
counts, and sets whose tiles all stay (a single basin with a wide k)."""
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

"""The trace contraction (data vectors and --nofit): sizes around the tiles
(128 x 128 frames, K-groups of 16 triples), lists that fill within a tile, and
the ordered self query with its band pass on both sides of 4096 vectors.
Distances are FP64 re-scores: the oracle's to rounding (1e-9 relative for
Euclidean distances), and equal bits between two routes of one query."""
import numpy as np
import pytest

import oracle
from mdsctk_amd import knn, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["bf16", "fp32"])
@pytest.mark.parametrize("n_ref,n_fit,vdim,k", [
    (33, 40, 1, 5), (127, 129, 47, 20), (128, 128, 48, 128), (129, 127, 49, 129),
    (260, 33, 145, 260), (3100, 2100, 24, 33), (9000, 700, 6, 255)])
def test_vectors_at_tile_edges(prec, n_ref, n_fit, vdim, k):
    ref = synth.data_vectors(n_ref, vdim, 1)
    fit = synth.data_vectors(n_fit, vdim, 2)
    with knn.KnnContext(0, prec) as ctx:
        ctx.set_data_reference(ref, "euclidean")
        d, i = ctx.data_query(fit, k)
    rows = np.arange(0, n_fit, max(1, n_fit // 40))
    d_o, _ = oracle.knn_data(ref, fit[rows], k, "euclidean")
    assert (np.abs(d[rows] - d_o) <= 1e-9 * np.maximum(1.0, d_o)).all()
    for r in rows:
        assert len(set(i[r].tolist())) == i.shape[1]
        own = np.sqrt(((fit[r] - ref[i[r]]) ** 2).sum(axis=1))
        assert (np.abs(d[r] - own) <= 1e-9 * np.maximum(1.0, own)).all()


@pytest.mark.parametrize("prec", ["bf16", "fp32"])
@pytest.mark.parametrize("metric", ["euclidean", "correlation"])
@pytest.mark.parametrize("kind", ["clusters", "dihedral", "offset"])
def test_vectors_against_themselves(prec, metric, kind):
    for n, k in ((4095, 30), (4096, 30), (4500, 5), (4609, 200)):
        x = synth.data_vectors(n, 45, 3, kind)
        out = []
        for sym in (1, 0):
            with knn.KnnContext(0, prec) as ctx:
                ctx.set_option(knn.OPT_SELF_SYMMETRIC, sym)
                ctx.set_data_reference(x, metric)
                out.append(ctx.data_query(None, k))
        np.testing.assert_array_equal(out[0][1], out[1][1])
        np.testing.assert_array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("prec", ["bf16", "fp16", "fp32"])
def test_frames_as_given_against_themselves(prec):
    x = synth.metastable_trajectory(4700, 33, 8, n_centres=9)
    x = (x - x.mean(axis=1, keepdims=True)).astype(np.float32)
    w = synth.masses(33, "random", 7)
    out = []
    for sym in (1, 0):
        with knn.KnnContext(0, prec) as ctx:
            ctx.set_option(knn.OPT_SELF_SYMMETRIC, sym)
            ctx.set_reference(x, w)
            out.append(ctx.query(None, 40, knn.KNN_NOFIT))
    np.testing.assert_array_equal(out[0][1], out[1][1])
    np.testing.assert_array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("power", [-60, 60])
def test_vectors_near_the_ends_of_the_range(power):
    """Scaling by a power of two scales every value, sum and distance exactly:
    the same rows at G terms around 1e-36 and 1e37."""
    x = synth.data_vectors(4300, 45, 3, "dihedral")
    out = []
    for f in (1.0, 2.0 ** power):
        with knn.KnnContext(0, "bf16") as ctx:
            ctx.set_data_reference(x * f, "euclidean")
            out.append(ctx.data_query(None, 20))
            out[-1] += ctx.data_query(x[:500] * f, 20)
    for j in (1, 3):
        np.testing.assert_array_equal(out[0][j], out[1][j])
    for j in (0, 2):
        np.testing.assert_array_equal(out[0][j] * 2.0 ** power, out[1][j])

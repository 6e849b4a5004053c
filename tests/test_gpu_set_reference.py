"""A resident set replaced by another of the same shape."""
import numpy as np
import pytest
import torch

from mdsctk_amd import knn, synth

pytestmark = pytest.mark.gpu


def test_device_frames_of_the_same_shape_wait_for_their_producer():
    """The second set's frames are still being written, by another stream's
    kernels, when the call that replaces the first set is made."""
    n, natoms, k = 2000, 100, 5
    first, second = synth.trajectory(n, natoms, 1), synth.trajectory(n, natoms, 2)
    fit = second[:50]
    buf = torch.from_numpy(first).cuda()
    late = torch.from_numpy(second).cuda()
    with knn.KnnContext(0, "bf16") as ctx:
        ctx.set_reference(second)
        want = ctx.query(fit, k)
        torch.cuda.synchronize()
        ctx.set_reference_device(buf.data_ptr(), n, natoms)
        torch.cuda._sleep(200_000_000)  # some 0.1 s
        buf.copy_(late)
        ctx.set_reference_device(buf.data_ptr(), n, natoms)
        got = ctx.query(fit, k)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(got[1], want[1])
    np.testing.assert_array_equal(got[0], want[0])


def test_host_frames_of_the_same_shape():
    """Buffers kept from one set to the next hold nothing of the last one:
    weights, --nofit operands and rows are the new set's."""
    n, natoms, k = 1300, 70, 6
    sets = [(synth.trajectory(n, natoms, s), synth.masses(natoms, "random", s)) for s in (3, 4)]
    fresh = []
    for x, w in sets:
        with knn.KnnContext(0, "bf16") as ctx:
            ctx.set_reference(x, w)
            fresh.append([ctx.query(None, k), ctx.query(x[:40], k, knn.KNN_NOFIT)])
    with knn.KnnContext(0, "bf16") as ctx:
        for (x, w), want in zip(sets * 2, fresh * 2):
            ctx.set_reference(x, w)
            for got, (d, i) in zip([ctx.query(None, k), ctx.query(x[:40], k, knn.KNN_NOFIT)], want):
                np.testing.assert_array_equal(got[1], i)
                np.testing.assert_array_equal(got[0], d)

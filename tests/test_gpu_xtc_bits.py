"""The device XTC reader's bit arithmetic against the host decoder, bit for
bit: packed triples of every width around 32, 64 and 72 bits (64-bit
reciprocals up to 64, a byte at a time beyond), per-axis widths, one-valued
axes, and frame counts on both sides of the frames-per-wave steps."""
import numpy as np
import pytest

from tests.test_formats import xtc_write
from tests.test_gpu_xtc import _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [1, 7, 10, 11, 15, 16, 20, 21, 22, 23, 24, 25])
@pytest.mark.parametrize("flat", [0, 1, 2])
def test_triple_widths(tmp_path, bits, flat):
    """Axes of `bits` bits each (25 and over take per-axis widths); flat axes
    hold one value."""
    rng = np.random.default_rng(bits + 40 * flat)
    x = rng.integers(0, 1 << bits, size=(37, 23, 3)).astype(np.float64)
    x[:, 0] = 0
    x[:, 1] = (1 << bits) - 1
    x[:, :, :flat] = 5
    # a coarse quantum keeps the values exact in float32
    f = str(tmp_path / "w.xtc")
    assert xtc_write(f, (x / 2.0).astype(np.float32), 2.0) == 0
    _same(f)


@pytest.mark.parametrize("n", [1, 7, 8, 9, 65, 16383, 16384, 33000])
def test_frames_per_wave(tmp_path, n):
    rng = np.random.default_rng(n)
    f = str(tmp_path / "n.xtc")
    assert xtc_write(f, rng.normal(size=(n, 11, 3)).astype(np.float32), 1000.0) == 0
    _same(f)

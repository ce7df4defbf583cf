"""Horizontal doubling where its one-pass kernels end: the smallest and largest
fixed lengths, a length of each kind per direction, line groups that do not
divide the box, a single plane; against the CPU oracle.

Tolerance: two FP64 transforms of at most 512 points per direction, each within
a few eps log2(n) of the norm of its line: 1e-12 of the largest value."""
import numpy as np
import pytest

from oracle import pyoracle

pytestmark = pytest.mark.gpu

# (nz, ny, nx)
SHAPES = [(2, 8, 8), (1, 256, 30), (3, 16, 512), (2, 512, 12), (2, 14, 32), (2, 32, 14), (5, 54, 120), (3, 22, 26)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_expand(shape):
    import fug30v0kxc_amd as fa
    print(f"[expand] {shape}", flush=True)
    a = np.random.RandomState(shape[1] + 3 * shape[2]).randn(*shape) + 2.0
    got = fa.expand(a)
    want = pyoracle.expand(a)
    assert got.shape == want.shape
    assert np.abs(got - want).max() < 1e-12 * np.abs(want).max()

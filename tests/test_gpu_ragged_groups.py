"""Boxes whose column pairs do not fill the y passes' groups (nx / 2 no multiple
of 4, 8 or 16), at y lengths of every group width, against the CPU oracle with
the tolerances of the operator and step tests."""
import numpy as np
import pytest

from oracle import pyoracle
from tests.test_gpu_fused_passes import NAMES, make_pair, rel

pytestmark = pytest.mark.gpu

SHAPES = [(30, 256, 6), (20, 512, 6), (4, 8, 8), (6, 64, 8), (18, 128, 7), (50, 60, 6), (90, 16, 6), (8, 160, 6),
          (14, 1024, 6)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_operators(shape):
    import fug30v0kxc_amd as fa
    print(f"[ragged] operators {shape}", flush=True)
    s, o = make_pair(*shape)
    f = np.random.RandomState(4).randn(*s.shape) + 3.0
    assert rel(s.d1bydy(f), o.d1bydy(f)) < 1e-12
    for a, b in zip(s.d2bydy(f), o.d2bydy(f)):
        assert rel(a, b) < 1e-12
    assert rel(s.dealias(f), o.dealias(f)) < 1e-13
    F = o.forwardfft(f)
    assert rel(s.forwardfft(f), F) < 1e-13
    assert rel(s.inversefft(F), o.inversefft(F)) < 1e-13
    assert rel(fa.expand(f), pyoracle.expand(f)) < 1e-12
    s.close()


@pytest.mark.parametrize("prec,tol", [(0, 1e-10), (1, 1e-5)], ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_steps(shape, prec, tol):
    print(f"[ragged] steps {shape} precision {prec}", flush=True)
    s, o = make_pair(*shape, prec=prec)
    s.step(12, 1e-6, 0)
    o.step(12, 1e-6, 0)
    for n in NAMES:
        assert rel(s.field(n), o[n]) < tol, n
    s.close()

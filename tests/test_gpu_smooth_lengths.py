"""The register-blocked kernels of the lengths that are multiples of 4 with
further factors 3 and 5 (36, 72, 100, 108, 144, 180, 200, 216), each along x and
along y, against the CPU oracle (tolerances of the operator and step tests)."""
import numpy as np
import pytest

from oracle import pyoracle
from tests.test_gpu_fused_passes import NAMES, make_pair, rel

pytestmark = pytest.mark.gpu

SHAPES = [(36, 72, 6), (72, 36, 7), (100, 108, 6), (108, 100, 6), (144, 180, 6), (180, 144, 6), (200, 216, 6),
          (216, 200, 6)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_operators(shape):
    import fug30v0kxc_amd as fa
    print(f"[lengths] operators {shape}", flush=True)
    s, o = make_pair(*shape)
    f = np.random.RandomState(4).randn(*s.shape) + 3.0
    for d1, d2 in (("d1bydx", "d2bydx"), ("d1bydy", "d2bydy")):
        assert rel(getattr(s, d1)(f), getattr(o, d1)(f)) < 1e-12
        for a, b in zip(getattr(s, d2)(f), getattr(o, d2)(f)):
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
    print(f"[lengths] steps {shape} precision {prec}", flush=True)
    s, o = make_pair(*shape, prec=prec)
    s.step(12, 1e-6, 0)
    o.step(12, 1e-6, 0)
    for n in NAMES:
        assert rel(s.field(n), o[n]) < tol, n
    s.close()

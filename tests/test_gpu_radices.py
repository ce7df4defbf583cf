"""The run-time radix transforms on lengths whose factors reach every butterfly
(2, 3, 4, 5, 7, 8, 11, 13) and the direct passes of larger primes, against the
CPU oracle (tolerances of the operator tests)."""
import numpy as np
import pytest

from oracle.pyoracle import Oracle
from tests.conftest import reference_params

pytestmark = pytest.mark.gpu

# 72 = 8 3 3, 98 = 2 7 7, 104 = 8 13, 110 = 2 5 11, 150 = 2 3 5 5, 288 = 8 4 3 3,
# 38 = 2 19, 1000 = 8 5 5 5, 2000 = 4 4 5 5 5, 18 = 2 3 3
SIZES = [(72, 98, 6), (104, 110, 6), (150, 38, 7), (1000, 18, 6), (18, 2000, 6), (288, 54, 6)]


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


@pytest.mark.parametrize("shape", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_operators(shape):
    from fug30v0kxc_amd import Solver
    nx, ny, nz = shape
    print(f"[radices] {shape}", flush=True)
    p = reference_params()
    s, o = Solver(nx, ny, nz, p), Oracle(nx, ny, nz, p)
    f = np.random.RandomState(4).randn(nz, ny, nx) + 3.0
    for d1, d2 in (("d1bydx", "d2bydx"), ("d1bydy", "d2bydy")):
        assert rel(getattr(s, d1)(f), getattr(o, d1)(f)) < 1e-12
        for a, b in zip(getattr(s, d2)(f), getattr(o, d2)(f)):
            assert rel(a, b) < 1e-12
    assert rel(s.dealias(f), o.dealias(f)) < 1e-13
    F = o.forwardfft(f)
    assert rel(s.forwardfft(f), F) < 1e-13
    assert rel(s.inversefft(F), o.inversefft(F)) < 1e-13
    s.close()

"""A state with content in the 2/3 band of pol and tor (set by the caller): the
step that follows reads it, the steps after that find the band zero again.
FP64 steps against the CPU oracle, tolerances of the step tests (1e-10; mixed
1e-5)."""
import numpy as np
import pytest

from tests.test_gpu_fused_passes import make_pair, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [(0, 1e-10), (1, 1e-5)], ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape", [(30, 30, 60), (64, 26, 13), (22, 64, 12), (8, 8, 6)],
                         ids=lambda s: "x".join(map(str, s)))
def test_band_content(shape, prec, tol):
    print(f"[band] {shape} precision {prec}", flush=True)
    s, o = make_pair(*shape, prec=prec)
    s.step(3, 1e-6, 0)
    o.step(3, 1e-6, 0)
    rng = np.random.RandomState(5)
    for n in ("pol", "tor"):
        o[n][:] = 1e-3 * rng.randn(*s.shape)
        s.set_field(n, o[n])
    for steps in (1, 2):
        s.step(steps, 1e-6, 0)
        o.step(steps, 1e-6, 0)
        for n in ("poldot", "tordot"):
            assert rel(s.field(n, 2), o[n][1]) < tol, n
        for n in ("pol", "tor", "bx", "by", "bz", "u", "w"):
            assert rel(s.field(n), o[n]) < tol, n
    s.close()

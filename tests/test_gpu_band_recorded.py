"""Recording an ensemble's steps leaves what is known of a box as it was: content
in the 2/3 band of pol and tor, set before, is still read by the box's own next
step.  FP64 (10 significant digits of the oracle, as in the step tests) and mixed
(1e-5)."""
import numpy as np
import pytest

from tests.test_gpu_fused_passes import make_pair, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [(0, 1e-10), (1, 1e-5)], ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape", [(30, 30, 20), (22, 64, 12)], ids=lambda s: "x".join(map(str, s)))
def test_band_content_over_a_recording(shape, prec, tol):
    print(f"[band, recorded] {shape} precision {prec}", flush=True)
    from fug30v0kxc_amd import Ensemble
    s, o = make_pair(*shape, prec=prec)
    s.step(4, 1e-6, 0)
    o.step(4, 1e-6, 0)
    rng = np.random.RandomState(5)
    for n in ("pol", "tor"):
        o[n][:] = 1e-3 * rng.randn(*s.shape)
        s.set_field(n, o[n])
    e = Ensemble([s], 1e-6)          # the box is past its start-up steps: none is taken
    s.step(1, 1e-6, 0)
    o.step(1, 1e-6, 0)
    for n in ("poldot", "tordot"):
        assert rel(s.field(n, 2), o[n][1]) < tol, n
    for n in ("pol", "tor", "bx", "by", "bz", "u", "w"):
        assert rel(s.field(n), o[n]) < tol, n
    e.close()
    s.close()

"""The right-hand sides at the register-blocked lengths from 480 points on, where
a full group of columns holds 4 pairs and the FP64 second derivatives and cross
products take 2: groups that a row fills (16 columns) and does not (10), and the
same lengths along x.  Against the CPU oracle with the tolerances of the routines'
tests (FP64 1e-11, mixed 1e-5)."""
import pytest

from tests.test_gpu_fused_passes import make_pair, rel

pytestmark = pytest.mark.gpu

SHAPES = [(nx, n, nz) for n in (480, 640, 768, 1024) for nx, nz in ((16, 6), (10, 7))]
SHAPES += [(480, 12, 6), (640, 6, 7)]


@pytest.mark.parametrize("prec,tol", [(0, 1e-11), (1, 1e-5)], ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_right_hand_sides(shape, prec, tol):
    print(f"[long] {shape} precision {prec}", flush=True)
    s, o = make_pair(*shape, prec=prec)
    s.hydro_deriv()
    o.hydro_deriv()
    for n in ("rdot", "tdot", "udot", "vdot", "wdot"):
        assert rel(s.field(n, 3), o[n][2]) < tol, n
    s.mag_deriv()
    o.mag_deriv()
    for n in ("poldot", "tordot"):
        assert rel(s.field(n, 3), o[n][2]) < tol, n
    s.close()

"""Steps and right-hand sides on lengths without a register-blocked plan (twice an
odd number, or a factor above 5), beyond the short ones: the run-time radix
kernels with auxiliary lines and two or three outputs, alone (both directions) and
beside a direction that has a plan, and one length per direction whose two-output
jobs need more than 64 KB of LDS.  Against the CPU oracle with the tolerances of the
routines' tests (FP64 1e-11, after steps 1e-10, mixed 1e-5)."""
import pytest

from tests.test_gpu_fused_passes import NAMES, make_pair, rel

pytestmark = pytest.mark.gpu

# 88 = 8 11, 84 = 4 3 7, 140 = 4 5 7, 102 = 2 3 17, 1400 = 8 5 5 7
SHAPES = [(88, 84, 9), (140, 88, 7), (84, 64, 8), (64, 140, 8), (102, 14, 10), (1400, 6, 6), (6, 1400, 6)]


@pytest.mark.parametrize("prec,tol", [(0, 1e-11), (1, 1e-5)], ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_right_hand_sides(shape, prec, tol):
    print(f"[no plan] right-hand sides {shape} precision {prec}", flush=True)
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


@pytest.mark.parametrize("prec,tol", [(0, 1e-10), (1, 1e-5)], ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape", SHAPES[:5], ids=lambda s: "x".join(map(str, s)))
def test_steps(shape, prec, tol):
    print(f"[no plan] steps {shape} precision {prec}", flush=True)
    s, o = make_pair(*shape, prec=prec)
    s.step(12, 1e-6, 0)
    o.step(12, 1e-6, 0)
    for n in NAMES:
        assert rel(s.field(n), o[n]) < tol, n
    s.close()

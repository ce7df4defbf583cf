"""The fused horizontal passes at the sizes where their tiles, plans and row
pairs end, against the CPU oracle: second derivatives with the Maxwell and
composite stresses as auxiliary lines, the EMF's x pass with the spectral
curl, bandj's x pass with and without the zero 2/3 band, the column kernels'
wall and short-walk launches, and boxes whose two horizontal lengths take
different kernels (register-blocked and run-time radices).

FP64 tolerances are those of the routines' own tests (1e-11 per routine,
1e-10 after steps); mixed ones the mode's 1e-5."""
import numpy as np
import pytest

from oracle.pyoracle import Oracle
from tests.conftest import reference_params

pytestmark = pytest.mark.gpu

NAMES = ("r", "t", "u", "v", "w", "bx", "by", "bz")
# (nx, ny, nz): plans with a radix 8 moved to the middle (120, 128, 160, 512) or
# first (32), one-pass and odd-radix plans (8, 30), line groups that do not
# divide the box, one length of each kind per direction, walls without
# interior planes (nz 6, 8) and with one (9)
SHAPES = [(160, 12, 9), (24, 128, 6), (120, 30, 8), (512, 8, 7), (8, 512, 6), (32, 20, 25), (30, 30, 60),
          (22, 64, 12), (64, 26, 13), (54, 18, 10)]


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


def make_pair(nx, ny, nz, prec=0, **kw):
    from fug30v0kxc_amd import Solver
    p = reference_params(b_amp=1e-2, **kw)
    o = Oracle(nx, ny, nz, p)
    o.setup_static()
    rng = np.random.RandomState(nx + 7 * ny)
    for n in ("u", "v", "w"):
        o[n][:] = 1e-2 * rng.randn(nz, ny, nx)
    o["w"][[0, -1]] = 0.0
    s = Solver(nx, ny, nz, p, precision=prec)
    s.set_state(*[o[n] for n in NAMES])
    return s, o


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_routines(shape):
    print(f"[fused] routines {shape}", flush=True)
    s, o = make_pair(*shape)
    s.hydro_deriv()
    o.hydro_deriv()
    for n in ("rdot", "tdot", "udot", "vdot", "wdot"):
        assert rel(s.field(n, 3), o[n][2]) < 1e-11, n
    s.mag_deriv()
    o.mag_deriv()
    for n in ("poldot", "tordot"):
        assert rel(s.field(n, 3), o[n][2]) < 1e-11, n
    # pol and tor with content in the 2/3 band: bandj on its own drops nothing
    rng = np.random.RandomState(3)
    for n in ("pol", "tor"):
        o[n][:] = rng.randn(*s.shape)
        s.set_field(n, o[n])
    s.bandj()
    o.bandj()
    for n in ("bx", "by", "bz", "jsq"):
        assert rel(s.field(n), o[n]) < 1e-11, n
    s.close()


@pytest.mark.parametrize("prec,tol", [(0, 1e-10), (1, 1e-5)], ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_steps(shape, prec, tol):
    # past the Euler and two-level start and one dealias (step 10), eta(z) on
    print(f"[fused] steps {shape} precision {prec}", flush=True)
    s, o = make_pair(*shape, prec=prec)
    s.step(12, 1e-6, 0)
    o.step(12, 1e-6, 0)
    for n in NAMES:
        assert rel(s.field(n), o[n]) < tol, n
    for n in ("bxbar", "bybar"):
        assert np.abs(s.field(n) - o[n]).max() <= tol * max(np.abs(o[n]).max(), 1e-6), n
    s.close()

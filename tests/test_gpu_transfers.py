"""State transfers large enough to be copied by several host threads: what is
set is what is read back, and the mixed mode's magnetic field is the FP32
fluctuation about its plane means."""
import numpy as np
import pytest

from tests.conftest import reference_params

pytestmark = pytest.mark.gpu

NAMES = ("r", "t", "u", "v", "w", "bx", "by", "bz")


@pytest.mark.parametrize("shape", [(256, 128, 129), (128, 96, 41), (30, 30, 7)], ids=lambda s: "x".join(map(str, s)))
def test_round_trip(shape):
    from fug30v0kxc_amd import MHD_PREC_MIXED, Solver
    nx, ny, nz = shape
    print(f"[transfers] {shape}", flush=True)
    rng = np.random.RandomState(6)
    st = {n: rng.randn(nz, ny, nx) + (3.0 if n in "rt" else 0.0) for n in NAMES}
    with Solver(nx, ny, nz, reference_params()) as s:
        s.set_state(**st)
        got = s.get_state()
        for n in NAMES:
            assert np.array_equal(got[n], st[n]), n
    with Solver(nx, ny, nz, reference_params(), precision=MHD_PREC_MIXED) as s:
        s.set_state(**st)
        got = s.get_state()
        bzbar = s.scalars()["bzbar"]
        assert abs(bzbar - st["bz"][0].mean()) < 1e-13
        mean = {"bx": s.field("bxbar")[:, None, None], "by": s.field("bybar")[:, None, None], "bz": bzbar}
        for n in ("r", "t", "u", "v", "w"):
            assert np.array_equal(got[n], st[n]), n
        # bxbar, bybar were cleared on the walls after the fluctuations were taken
        for n in ("bx", "by", "bz"):
            want = np.float32(st[n] - (st[n].mean((1, 2), keepdims=True) if n != "bz" else bzbar)) + mean[n]
            assert np.abs(got[n] - want).max() < 1e-6, n

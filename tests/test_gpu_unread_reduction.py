"""A reduction whose result nobody asks for (mhd_global_averages without `out`)
returns before it has run; a field set right after it arrives whole, and the next
reduction's result is its own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "mixed"])
def test_field_set_behind_an_unread_reduction(prec):
    print(f"[unread reduction] precision {prec}", flush=True)
    from fug30v0kxc_amd import Solver, reference_params
    nx, ny, nz = 128, 96, 64
    s = Solver(nx, ny, nz, reference_params(t_amp=1e-3), prec)
    s.static()
    rng = np.random.RandomState(3)
    for _ in range(8):
        f = rng.standard_normal((nz, ny, nx))
        f[0, 0, :8] = 1e3 + np.arange(8)
        assert s._lib.mhd_global_averages(s._ctx, None) == 0
        s.set_field("w", f)
        assert np.array_equal(s.field("w"), f)
        assert s._lib.mhd_global_averages(s._ctx, None) == 0
        assert s.sminmax("w") == (f.min(), f.max())
    s.close()

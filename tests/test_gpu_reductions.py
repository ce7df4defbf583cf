"""The reductions over planes at the plane counts where their finishing kernel's
batches (8 planes, 64 lanes) end, against the CPU oracle with the tolerances of
test_gpu_physics."""
import numpy as np
import pytest

from tests.test_gpu_fused_passes import make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [6, 8, 9, 63, 64, 65, 130])
def test_reductions(nz):
    print(f"[reductions] 10x8x{nz}", flush=True)
    s, o = make_pair(10, 8, nz)
    assert abs(s.nusselt() - o.nusselt()) < 1e-12 * max(1.0, abs(o.nusselt()))
    assert np.allclose(s.checkdivb(), o.checkdivb(), rtol=1e-10, atol=1e-10)
    for n in ("t", "u", "w", "bz"):
        assert np.allclose(s.sminmax(n), o.sminmax(o[n]), rtol=1e-14, atol=0)
    assert abs(s.calcdt() - o.calcdt()) < 1e-14 * o.calcdt()
    assert np.allclose(s.GlobalAverages(), o.global_averages(), rtol=1e-11, atol=1e-18)
    s.close()

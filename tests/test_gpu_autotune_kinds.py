"""The autotuner times the launches that a box's step makes: choices for kinds the
step does not run stay as the caller set them, and every plan a caller may set is
right for the launches that the step runs with it (the EMF's cross product, the
inverse transform with two outputs, second derivatives with auxiliary lines), at
all lengths that have alternatives.  Tolerances of the step tests."""
import numpy as np
import pytest

from tests.test_gpu_fused_passes import NAMES, make_pair, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "mixed"])
def test_kinds_the_step_does_not_run_keep_their_choice(prec):
    print(f"[autotune] kept kinds, precision {prec}", flush=True)
    s, o = make_pair(64, 128, 16, prec=prec)
    s.set_tune(variant_x=[0, 0, 1, 1], variant_y=0, mult_x=[1, 1, 5, 7], mult_y=1, zc=8)
    t = s.autotune()
    assert t["variant_x"][2:] == [1, 1] and t["mult_x"][2:] == [5, 7]
    assert all(m in (1, 2) for m in t["mult_x"][:2] + t["mult_y"])
    # tuning between steps changes nothing but the rounding
    s.step(4, 1e-6, 0)
    o.step(4, 1e-6, 0)
    for n in NAMES:
        assert rel(s.field(n), o[n]) < (1e-5 if prec else 1e-10), n
    s.close()


def test_a_box_without_a_field_keeps_the_half_transforms():
    from fug30v0kxc_amd import Solver, reference_params
    p = reference_params(t_amp=1e-3)
    p["f"] = 0.0
    s = Solver(64, 64, 12, p)
    s.static()
    s.set_tune(variant_y=[0, 0, 1, 1], mult_y=[1, 1, 3, 4])
    t = s.autotune()
    assert t["variant_y"][2:] == [1, 1] and t["mult_y"][2:] == [3, 4]
    s.close()


@pytest.mark.parametrize("prec,tol", [(0, 1e-10), (1, 1e-5)], ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape", [(64, 160, 8), (160, 128, 6), (128, 512, 6), (512, 64, 6), (10, 256, 7), (256, 12, 7)],
                         ids=lambda s: "x".join(map(str, s)))
def test_steps_with_alternative_plans(shape, prec, tol):
    print(f"[autotune] plans {shape} precision {prec}", flush=True)
    s, o = make_pair(*shape, prec=prec)
    alt = lambda n: {256: 2, 10: 0, 12: 0}.get(n, 1)  # noqa: E731
    s.set_tune(variant_x=alt(shape[0]), variant_y=alt(shape[1]), mult_x=2, mult_y=1, zc=8)
    s.step(12, 1e-6, 0)
    o.step(12, 1e-6, 0)
    for n in NAMES:
        assert rel(s.field(n), o[n]) < tol, n
    s.close()

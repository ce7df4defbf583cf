"""checkdivb of a mixed-precision box.

The three derivatives of B are FP32 there and nearly cancel in a real field, so
the extremes of div B, handed out as 64-bit numbers, carry FP32 rounding.  Two
things are held: the digits themselves (one order of operations per length,
whatever plan the other passes of a box run; a change of that order moves the
extremes by 1e-8 and more, the bound here is 1e-10), and their distance from div
B of the same field in FP64.  That field is random, its derivatives do not
cancel: with eps = 2^-24 the FP32 field and a transform pair of length N give at
most about eps (2 log2 N + 4) of the largest derivative; the sum of three takes
the same factor, so 64 eps of max |div B| covers N up to 300.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (nx, ny, nz) -> max, min of div B of field(shape), as this order gives them
PINS = {
    (36, 30, 24): ("0x1.10d057a000000p+5", "-0x1.13d1a15000000p+5"),
    (72, 44, 33): ("0x1.b49d808000000p+5", "-0x1.ce06e3c000000p+5"),
    (100, 144, 20): ("0x1.d96db38000000p+5", "-0x1.d890ff0000000p+5"),
    (108, 180, 12): ("0x1.d6b6530400000p+5", "-0x1.b67e8b0000000p+5"),
    (200, 216, 10): ("0x1.4981f57000000p+6", "-0x1.3d98acd000000p+6"),
    (98, 242, 12): ("0x1.26f33e4800000p+6", "-0x1.33e1f88000000p+6"),
    (34, 286, 9): ("0x1.24a3d46000000p+6", "-0x1.2024f0c000000p+6"),
    (62, 26, 40): ("0x1.e8732dd000000p+5", "-0x1.0223458800000p+6"),
    (54, 250, 11): ("0x1.01b7db0000000p+6", "-0x1.12df819000000p+6"),
    (64, 48, 32): ("0x1.978d2a0000000p+5", "-0x1.976cf48000000p+5"),
    (30, 96, 13): ("0x1.e61f861000000p+4", "-0x1.e61d85c000000p+4"),
}


def field(shape):
    """B of order 0.1 with a mean field along z, exact in FP32 steps of 2^-20."""
    rng = np.random.RandomState(sum(shape))
    b = [rng.randint(-1 << 18, 1 << 18, shape) / float(1 << 20) for _ in range(3)]
    b[2] += 1.0
    return b


def solver(nx, ny, nz, prec):
    from fug30v0kxc_amd import Solver, reference_params
    s = Solver(nx, ny, nz, reference_params(ra=1e5, q=100.0), prec)
    shape = (nz, ny, nx)
    t = np.ones(shape) * np.linspace(1.0, 11.0, nz)[:, None, None]
    z = np.zeros(shape)
    s.set_state(t, t, z, z, z, *field(shape))
    return s


@pytest.mark.parametrize("shape", list(PINS), ids=lambda s: "x".join(map(str, s)))
def test_mixed_checkdivb(shape):
    print(f"[mixed divb] {shape}", flush=True)
    from fug30v0kxc_amd import MHD_PREC_FP64, MHD_PREC_MIXED
    s = solver(*shape, MHD_PREC_MIXED)
    got = s.checkdivb()
    s.close()
    e = solver(*shape, MHD_PREC_FP64)
    exact = e.checkdivb()
    e.close()
    scale = max(abs(x) for x in exact)
    for g, p, x in zip(got, PINS[shape], exact):
        assert abs(g - x) <= 64 * 2.0 ** -24 * scale, (g, x)
        assert abs(g - float.fromhex(p)) <= 1e-10 * abs(g), (g.hex(), p)

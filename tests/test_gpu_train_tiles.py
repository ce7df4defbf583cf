"""The training kernel where its tiles of 32 cells end, and the update fused
into its reduction.

Tolerances: the gradient as in test_gpu_closure (bf16 operands, FP32 sums); the
update is FP32 arithmetic of a few operations on the same gradient, 1e-5 of lr."""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests.test_gpu_closure import F, _f32, _params

pytestmark = pytest.mark.gpu


def _closure(fields, shape):
    import fug30v0kxc_amd as fa
    cl = fa.Closure(seed=3)
    rng = np.random.default_rng(8)
    coarse = _f32({n: fields(rng, shape) for n in F})
    t = [np.asarray(0.5 * fields(rng, shape), np.float32).astype(np.float64) for _ in range(12)]
    cl.add(coarse, t)
    cl.norm = np.concatenate([np.zeros(8), np.ones(8), np.zeros(12), np.ones(12)])
    cl.params = _params(5, 0.2)
    return cl, coarse, t


@pytest.mark.parametrize("ncell", [8, 31, 33, 64, 1000])
def test_gradient_tiles(ncell):
    print(f"[train] gradient ncell={ncell}", flush=True)
    shape = (6, 8, 10)
    cl, coarse, t = _closure(lambda r, s: r.standard_normal(s), shape)
    cells = np.random.default_rng(ncell).integers(0, int(np.prod(shape)), size=ncell)
    Lg, gg = cl.grad(cells)
    Lo, go = po.mlp_grad([(coarse, t)], _params(5, 0.2).astype(np.float64), cl.norm, cells, round_bf16=True)
    assert abs(Lg - Lo) <= 1e-4 * Lo
    offs = [0, 13824, 13888, 17984, 18048, 18816, 18828]
    for a, b in zip(offs[:-1], offs[1:]):
        assert np.linalg.norm(gg[a:b] - go[a:b]) < 1e-2 * np.linalg.norm(go[a:b]), a


@pytest.mark.parametrize("batch", [32, 96, 4096])
def test_update_is_adam_of_the_gradient(batch):
    # every cell of the data set is alike, so any sample has the same gradient
    print(f"[train] update batch={batch}", flush=True)
    cl, _, _ = _closure(lambda r, s: np.full(s, r.standard_normal()), (5, 6, 8))
    m = v = np.zeros(po.N_PARAM, np.float32)
    lr = 1e-3
    for t in (1, 2, 3):
        p = cl.params.astype(np.float32)
        _, g = cl.grad(np.zeros(batch, np.int64))
        cl.train(1, batch=batch, lr=lr)
        m = np.float32(0.9) * m + np.float32(0.1) * g
        v = np.float32(0.999) * v + np.float32(0.001) * g * g
        mh, vh = m / np.float32(1 - 0.9 ** t), v / np.float32(1 - 0.999 ** t)
        want = p - np.float32(lr) * mh / (np.sqrt(vh) + np.float32(1e-8))
        assert np.abs(cl.params - want).max() <= 1e-5 * lr + 1.2e-7 * np.abs(p).max(), t

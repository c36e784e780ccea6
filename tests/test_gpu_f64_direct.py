"""Small fp64 products (gemm_f64_direct_kernel, 16 x 16 and 32 x 32 tiles, K
dealt over the waves): tile edges and K around a block of 32 and the four waves'
share, in every layout, with accumulation.  Bar: K 2^-53 (|A| |B|), the bound of
a sum of K products in any order, and exactness on integers."""
import numpy as np
import pytest
import torch

import momijo_amd as mj
from _util import to_dev

pytestmark = pytest.mark.gpu


def _view(t, layout):
    if layout == "n":
        return t.contiguous()
    if layout == "t":
        return t.t().contiguous().t()
    wide = torch.zeros((t.shape[0], 2 * t.shape[1] + 1), dtype=t.dtype, device=t.device)
    view = wide[:, 1::2]
    view.copy_(t)
    return view


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (16, 16, 32), (17, 33, 31), (33, 15, 127), (70, 59, 129),
                                   (59, 70, 1779), (300, 200, 260), (400, 490, 161), (512, 512, 65), (513, 480, 65)])
@pytest.mark.parametrize("la,lb", [("n", "t"), ("n", "n"), ("t", "n"), ("t", "t"), ("s", "n")])
def test_layouts(dev, M, N, K, la, lb):
    rng = np.random.default_rng(M + 3 * N + 7 * K)
    a, b = rng.standard_normal((M, K)), rng.standard_normal((K, N))
    got = mj.matmul(mj.Tensor(_view(to_dev(a, dev), la)), mj.Tensor(_view(to_dev(b, dev), lb)))
    ref = a.astype(np.longdouble) @ b.astype(np.longdouble)
    bound = K * 2.0 ** -53 * (np.abs(a) @ np.abs(b))
    assert np.all(np.abs(got.numpy() - ref) <= bound)
    ai, bi = rng.integers(-99, 100, (M, K)), rng.integers(-99, 100, (K, N))
    got = mj.matmul(mj.Tensor(_view(to_dev(ai.astype(np.float64), dev), la)),
                    mj.Tensor(_view(to_dev(bi.astype(np.float64), dev), lb)))
    np.testing.assert_array_equal(got.numpy(), (ai @ bi).astype(np.float64))


def test_accumulation(dev):
    rng = np.random.default_rng(5)
    a, b, g = (rng.integers(-99, 100, s).astype(np.float64) for s in ((90, 300), (300, 70), (90, 70)))
    ga0, gb0 = rng.integers(-9, 10, a.shape).astype(np.float64), np.ones_like(b)
    t = lambda x: mj.Tensor(to_dev(x, dev))  # noqa: E731
    ga, gb = mj.matmul_backward(t(a), t(b), t(g), t(ga0), t(gb0))
    np.testing.assert_array_equal(ga.numpy(), ga0 + g @ b.T)
    np.testing.assert_array_equal(gb.numpy(), gb0 + a.T @ g)

"""The tiny fp32 products (gemm_f32_tiny_kernel: 16 x 16 and 32 x 32 tiles, K in
rounds of 256): tile edges, K around a round and off multiples of 4, every
layout and both gradients' accumulation.  Bar against the strict-order fp32
recurrence: 2 K 2^-24 (|A| |B|), K roundings of at most 2^-24 of the absolute
sum on either side; all layouts give the same bits."""
import numpy as np
import pytest
import torch

import momijo_amd as mj
from _util import to_dev

pytestmark = pytest.mark.gpu

_SHAPES = [(1, 1, 1), (16, 16, 256), (17, 15, 257), (31, 33, 255), (250, 3, 1000), (1, 1000, 1024),
           (256, 256, 256), (100, 500, 300), (33, 400, 513), (512, 440, 70)]


def _strict(a, b):
    """The fp32 sums in ascending k, one rounding per product."""
    acc = np.zeros((a.shape[0], b.shape[1]), np.float32)
    for k in range(a.shape[1]):
        acc = (acc.astype(np.float64) + np.outer(a[:, k].astype(np.float64), b[k])).astype(np.float32)
    return acc


def _view(t, layout):
    if layout == "n":
        return t.contiguous()
    if layout == "t":
        return t.t().contiguous().t()
    wide = torch.zeros((t.shape[0], 2 * t.shape[1] + 1), dtype=t.dtype, device=t.device)
    view = wide[:, 1::2]
    view.copy_(t)
    return view


@pytest.mark.parametrize("M,N,K", _SHAPES)
def test_strict_order_in_every_layout(dev, M, N, K):
    rng = np.random.default_rng(M + 3 * N + 7 * K)
    a = rng.standard_normal((M, K)).astype(np.float32)
    b = rng.standard_normal((K, N)).astype(np.float32)
    want = _strict(a, b)
    ta, tb = to_dev(a, dev), to_dev(b, dev)
    first = None
    for la, lb in (("n", "t"), ("n", "n"), ("t", "n"), ("t", "t"), ("s", "n"), ("n", "s")):
        got = mj.matmul(mj.Tensor(_view(ta, la)), mj.Tensor(_view(tb, lb))).torch
        if first is None:
            first = got
            bound = 2 * K * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b))
            assert np.all(np.abs(got.cpu().numpy().astype(np.float64) - want) <= bound)
        assert torch.equal(got, first), (la, lb)


def test_batches_and_accumulation(dev):
    rng = np.random.default_rng(3)
    a = rng.integers(-8, 9, size=(3, 1, 20, 37)).astype(np.float32)
    b = rng.integers(-8, 9, size=(2, 37, 19)).astype(np.float32)
    got = mj.tensordot(mj.Tensor(to_dev(a, dev)), mj.Tensor(to_dev(b, dev))).numpy()
    np.testing.assert_array_equal(got, (a.astype(np.float64) @ b).astype(np.float32))
    ctx = mj.GradContext()
    x = rng.integers(-8, 9, size=(40, 23)).astype(np.float32)
    w = rng.integers(-8, 9, size=(23, 50)).astype(np.float32)
    gx = mj.GradTensor.from_tensor(ctx, mj.Tensor(to_dev(x, dev)), True)
    gw = mj.GradTensor.from_tensor(ctx, mj.Tensor(to_dev(w, dev)), True)
    y = gx.matmul2d(ctx, gw)
    y.backward(ctx)
    y.backward(ctx)    # a second pass adds onto the first's gradients
    ones = np.ones((40, 50), np.float32)
    np.testing.assert_array_equal(gx.grad(ctx).numpy(), 2 * (ones @ w.T))
    np.testing.assert_array_equal(gw.grad(ctx).numpy(), 2 * (x.T @ ones))

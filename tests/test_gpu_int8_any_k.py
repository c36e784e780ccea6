"""int8 products whose rows start at any byte (K not a multiple of 16, or an
unaligned operand): exact int32 sums at tile edges (64 x 64, 128 x 128) and K
around a 16-byte chunk and a 64-deep stage, and QuantLinear on them."""
import numpy as np
import pytest
import torch

import momijo_amd as mj
from momijo_amd import _lib
from _util import to_dev

pytestmark = pytest.mark.gpu

_SHAPES = [(1, 1, 1), (3, 5, 15), (64, 64, 17), (65, 63, 63), (70, 130, 65), (2, 1856, 1015),
           (746, 19, 968), (300, 200, 129), (2100, 2049, 130)]


@pytest.mark.parametrize("M,N,K", _SHAPES)
def test_exact_sums(dev, M, N, K):
    rng = np.random.default_rng(M + 3 * N + 7 * K)
    a = rng.integers(-128, 128, size=(M, K)).astype(np.int8)
    w = rng.integers(-128, 128, size=(N, K)).astype(np.int8)
    got = mj.matmul_i8_i8_to_i32(mj.Tensor(to_dev(a, dev)),
                                 mj.Tensor(to_dev(w, dev)).transpose()).numpy()
    want = (a.astype(np.float64) @ w.astype(np.float64).T).astype(np.int32)  # |sum| < 2^24
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("shift", [1, 2, 4, 8])
def test_unaligned_operands(dev, shift):
    M, N, K = 130, 70, 96
    rng = np.random.default_rng(shift)
    a = rng.integers(-128, 128, size=M * K).astype(np.int8)
    w = rng.integers(-128, 128, size=N * K).astype(np.int8)
    ad = torch.zeros(M * K + shift, dtype=torch.int8, device=dev)
    wd = torch.zeros(N * K + 3 * shift, dtype=torch.int8, device=dev)
    ad[shift:] = to_dev(a, dev)
    wd[3 * shift:] = to_dev(w, dev)
    c = torch.empty((M, N), dtype=torch.int32, device=dev)
    _lib.call("mj_matmul_i8_i8_to_i32", ad.data_ptr() + shift, wd.data_ptr() + 3 * shift,
              c.data_ptr(), M, N, K, 0, torch.cuda.current_stream().cuda_stream)
    want = a.reshape(M, K).astype(np.int64) @ w.reshape(N, K).astype(np.int64).T
    np.testing.assert_array_equal(c.cpu().numpy(), want)


@pytest.mark.parametrize("M,N,K", [(33, 70, 31), (200, 300, 1001)])
def test_quant_linear(oracle, dev, M, N, K):
    x = oracle.randn_f32((M, K), seed=M)
    q = np.random.default_rng(N).integers(-127, 128, size=(N, K)).astype(np.int8)
    b = oracle.randn_f32((N,), seed=N)
    layer = mj.QuantLinear(K, N, mj.Tensor(to_dev(q, dev)), mj.Tensor(to_dev(b, dev)), 0.01, 0.03)
    got = layer.forward(mj.Tensor(to_dev(x, dev))).numpy()
    np.testing.assert_array_equal(got, oracle.quant_linear_fw(x, q, b, 0.01, 0.03))

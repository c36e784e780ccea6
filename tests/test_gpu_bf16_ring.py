"""The bf16 NT GEMM's ring tiles (32 x 32, 64 x 64, 128 x 64): tile edges, K
below and above the ring's depth, odd leading dimensions, against exact sums
(small integers: any order gives the same fp32 sum) and the oracle's bf16
rounding of them; capture stays refused by shape."""
import numpy as np
import pytest
import torch

import momijo_amd as mj
from _util import bf16_dev, bf16_host_bits, to_dev

pytestmark = pytest.mark.gpu

# M, N, K on: 32 x 32 (one workgroup, ragged; 4 per CU), 64 x 64 of five stages
# and of three, 128 x 64; K of 1 to many 64-deep stages, remainders of 8
_SHAPES = [(1, 1, 8), (33, 31, 56), (85, 16, 704), (65, 97, 328), (500, 2040, 64),
           (1000, 1030, 1024), (1024, 1024, 1096), (1000, 3000, 200), (1500, 1500, 648),
           (2048, 2048, 264), (2049, 2050, 2056), (512, 33, 3520), (1000, 1000, 4096)]


@pytest.mark.parametrize("M,N,K", _SHAPES)
@pytest.mark.parametrize("epi,pad", [(mj.EPI_NONE, 0), (mj.EPI_RELU, 8)])
def test_integer_exact(oracle, dev, M, N, K, epi, pad):
    rng = np.random.default_rng(M + 3 * N + 7 * K + pad)
    a = rng.integers(-3, 4, size=(M, K)).astype(np.float32)
    w = rng.integers(-3, 4, size=(N, K)).astype(np.float32)
    b = rng.integers(-8, 9, size=N).astype(np.float32)
    ad = torch.zeros((M, K + pad), dtype=torch.bfloat16, device=dev)[:, :K]
    ad.copy_(to_dev(a, dev))
    wd = bf16_dev(oracle.f32_to_bf16(w), dev)
    out = torch.zeros((M, N + pad), dtype=torch.bfloat16, device=dev)
    got = mj.gemm_bf16_nt(ad, wd, to_dev(b, dev), epi, out=out[:, :N])
    want = a.astype(np.float64) @ w.astype(np.float64).T + b
    if epi == mj.EPI_RELU:
        want = np.maximum(want, 0)
    np.testing.assert_array_equal(bf16_host_bits(got.contiguous()),
                                  oracle.f32_to_bf16(want.astype(np.float32)))
    if pad:
        assert not bool(out[:, N:].any())      # nothing written past the row


@pytest.mark.parametrize("M,N,K,taken", [(512, 512, 512, True), (1000, 1000, 4096, False)])
def test_capture_rule_by_shape(dev, M, N, K, taken):
    """Shapes that need no K split can be captured and replayed; shapes whose
    tiles split K stay refused under capture."""
    a = torch.randn((M, K), device=dev).bfloat16()
    w = torch.randn((N, K), device=dev).bfloat16()
    out = torch.empty((M, N), dtype=torch.bfloat16, device=dev)
    want = mj.gemm_bf16_nt(a, w).clone()
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        g.capture_begin()
        try:
            if taken:
                mj.gemm_bf16_nt(a, w, out=out)
            else:
                with pytest.raises(mj.MomijoHipError):
                    mj.gemm_bf16_nt(a, w, out=out)
        finally:
            g.capture_end()
    if taken:
        for _ in range(3):
            out.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)


def test_capture_refusal_names_its_reason(dev):
    """A shape refused for its own sake (its ring tile needs no workspace) is not
    told that it needs one."""
    a = torch.randn((1000, 4096), device=dev).bfloat16()
    w = torch.randn((1000, 4096), device=dev).bfloat16()
    out = torch.empty((1000, 1000), dtype=torch.bfloat16, device=dev)
    mj.gemm_bf16_nt(a, w, out=out)
    torch.cuda.synchronize()
    s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        g.capture_begin()
        try:
            with pytest.raises(mj.MomijoHipError, match="goes by the shape") as e:
                mj.gemm_bf16_nt(a, w, out=out)
        finally:
            g.capture_end()
    assert "this call needs" not in str(e.value) and "graph capture" in str(e.value)

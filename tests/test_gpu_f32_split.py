"""The fp32 products on split bf16 operands (gemm_f32s.hip): every kernel that
the launcher picks, at tile edges and K remainders, in all operand layouts;
and the values the split does not hold (infinities, NaN, magnitudes that round
to infinity in bf16, rows of tiny and denormal numbers).

Accuracy bar: the 2-norm of the error against the exact (64-bit) product,
relative to the product's, stays below 2^-24 sqrt(nk + 2) for nk blocks of 32
k.  Each block's sum and each of the nk additions onto the running sum rounds
by at most 2^-24 of a partial sum no larger (2-norm, independent terms) than
the result, and independent roundings add in squares.  Leaving out any of the
split's terms gives at least 2^-18; the native fp32 chain, K roundings, is
above the bar from K ~ 1000 on.
"""
import math

import numpy as np
import pytest
import torch

import momijo_amd as mj


def _plan(M, N, K, batches=1):
    """plan_f32s (gemm_f32s.hip); test_kernel_choice compares it with the library's."""
    nk = -(-K // 32)

    def tiles(tm, tn):
        return (-(-M // tm)) * (-(-N // tn)) * batches

    def tile_us(tm, tn, fixed, stage):
        return math.ceil(tiles(tm, tn) / 256) * (fixed + nk * stage)

    def direct_us(tb, nw, wait, work):
        return math.ceil(nk / (2 * nw)) * (wait + work * tiles(tb, tb) / 256)

    us = [tile_us(256, 128, 14, 2.45), tile_us(128, 128, 9, 1.35),
          tile_us(64, 64, 2.5, 0.45) + (0.12 * nk if tiles(64, 64) <= 256 else 0),
          direct_us(32, 4, 1.3, 1.6), direct_us(16, 4, 0.8, 0.9), direct_us(16, 16, 1.0, 4.3)]
    names = ["256x128", "128x128", "64x64", "direct32", "direct16", "direct16w16"]
    return names[us.index(min(us))]


# M, N, K above 256^3 multiply-adds or K above 1024: remainders of every tile dimension and of
# the 32-deep stage, K below one, two and three stages (and one below 17, on the native tiles)
_SHAPES = [(4095, 4097, 70), (4096, 4096, 288), (2049, 2000, 257), (2048, 2048, 96),
           (1000, 1030, 513), (1025, 1024, 31), (4099, 4093, 3), (2111, 2017, 33),
           (300, 517, 257), (515, 257, 1000), (33, 1000, 1030), (1, 4111, 4097), (4099, 1, 4113),
           (17, 301, 4100), (5, 9, 1025), (16, 16, 2048)]


def test_shapes_reach_every_kernel():
    assert {_plan(*s) for s in _SHAPES} == {"256x128", "128x128", "64x64", "direct32", "direct16",
                                            "direct16w16"}


def _view(t, layout):
    """The same values as row-major ("n"), as the transpose view of a row-major
    matrix ("t"), or as a view with both strides above one ("s")."""
    if layout == "n":
        return t.contiguous()
    if layout == "t":
        return t.t().contiguous().t()
    wide = torch.zeros((t.shape[0], 2 * t.shape[1] + 1), dtype=t.dtype, device=t.device)
    view = wide[:, 1::2]
    view.copy_(t)
    return view


def _check(got, a, b):
    ref = a.double() @ b.double()
    nk = -(-a.shape[1] // 32)
    err = float((got.double() - ref).norm() / ref.norm())
    assert err <= 2.0 ** -24 * math.sqrt(nk + 2), err


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", _SHAPES)
def test_layouts_and_accuracy(dev, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + 3 * N + 7 * K)
    a = torch.randn((M, K), generator=g, device=dev)
    b = torch.randn((K, N), generator=g, device=dev)
    want = None
    for la, lb in (("n", "t"), ("n", "n"), ("t", "n"), ("t", "t"), ("s", "n"), ("n", "s")):
        got = mj.matmul(mj.Tensor(_view(a, la)), mj.Tensor(_view(b, lb))).torch
        if want is None:
            _check(got, a, b)
            want = got
        assert torch.equal(got, want), (la, lb)   # one summation order for all


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(256, 292, 260), (1030, 1000, 257), (2049, 2000, 96),
                                   (4100, 4096, 64), (1, 4111, 4097)])
def test_values_outside_the_split(dev, M, N, K):
    """Rows and columns with special values give what fp32 gives: infinities
    and NaN where the exact product has them, values above bf16's largest
    finite number and rows of tiny or denormal numbers at fp32 accuracy; the
    other outputs are those of the same product without the special rows."""
    g = torch.Generator(device="cuda").manual_seed(K)
    a = torch.randn((M, K), generator=g, device=dev)
    b = torch.randn((K, N), generator=g, device=dev)
    plain = mj.matmul(mj.Tensor(a), mj.Tensor(b)).torch
    inf = float("inf")
    rows = sorted({0, M // 2, M - 1})
    for case in ("inf", "nan", "huge", "tiny", "denormal", "tinycol"):
        x, w = a.clone(), b.clone()
        cols = []
        if case == "inf":
            x[rows, K // 3] = inf
        elif case == "nan":
            x[rows, K - 1] = float("nan")
        elif case == "huge":
            x[rows, :] = 0.0
            x[rows, K // 2] = 3.4e38        # rounds to infinity in bf16
            w[K // 2, :] = w[K // 2, :].clamp(-1.0, 1.0) * 0.5
        elif case == "tiny":
            x[rows, :] *= 2.0 ** -115
        elif case == "denormal":
            x[rows, :] *= 2.0 ** -140       # Float32 denormals
        else:
            cols = sorted({0, N // 2, N - 1})
            w[:, cols] *= 2.0 ** -115
        got = mj.matmul(mj.Tensor(x), mj.Tensor(w)).torch
        ref = x.double() @ w.double()
        sel = got[rows] if not cols else got[:, cols]
        want = ref[rows] if not cols else ref[:, cols]
        if case == "inf":
            assert torch.equal(sel, want.float())
        elif case == "nan":
            assert torch.isnan(sel).all()
        else:
            # native fp32 sums: each of the K steps rounds by at most 2^-24 of a
            # partial sum no larger than the absolute sum, or by 2^-149 among
            # denormals
            absum = x.double().abs() @ w.double().abs()
            absum = absum[rows] if not cols else absum[:, cols]
            ok = (sel.double() - want).abs() <= K * (2.0 ** -24 * absum + 2.0 ** -149)
            assert bool(ok.all()), case
            if case in ("tiny", "tinycol"):
                assert float((sel.double() - want).norm() / want.norm()) <= 2.0 ** -24 * math.sqrt(K)
        keep = torch.ones_like(got, dtype=torch.bool)
        keep[rows if not cols else slice(None), :] = bool(cols)
        if cols:
            keep[:, cols] = False
        if case != "huge":
            assert torch.equal(got[keep], plain[keep]), case


@pytest.mark.gpu
def test_conv2d_values_outside_the_split(dev):
    """An infinity in the image reaches exactly the outputs whose window holds
    it; the rest keep their bits."""
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn((3, 40, 27, 31), generator=g, device=dev)
    conv = mj.Conv2d(40, 70, (3, 3), (1, 1), (1, 1))
    y0 = conv.forward(mj.Tensor(x)).torch
    x2 = x.clone()
    x2[1, 2, 5, 6] = float("inf")
    y1 = conv.forward(mj.Tensor(x2)).torch
    ref = torch.nn.functional.conv2d(x2.cpu().double(), conv.weight.torch.cpu().double(),
                                     padding=1).to(dev)
    hit = ~torch.isfinite(ref)
    assert hit.any() and torch.equal(y1[hit].double(), ref[hit])
    assert torch.equal(y1[~hit], y0[~hit])


def test_three_bf16_parts_hold_a_float32():
    """x = h + m + l exactly for 24-bit significands down to 2^-96 (CPU model
    of the split)."""
    rng = np.random.default_rng(1)
    x = (rng.standard_normal(100000) * 2.0 ** rng.integers(-90, 100, 100000)).astype(np.float32)
    t = torch.from_numpy(x)
    h = t.bfloat16().float()
    m = (t - h).bfloat16().float()
    l = (t - h - m).bfloat16().float()
    assert torch.equal(h.double() + m.double() + l.double(), t.double())


def test_conv_tap_division_by_reciprocal():
    """The conv gather's k / (kH kW) and t / kW by multiplied reciprocals: exact
    for every k that its tiles meet (K up to 2^26, the last stage up to 31 past
    it) and every tap of kernels up to 64 taps."""
    top = (1 << 26) + 32
    rng = np.random.default_rng(2)
    k = np.concatenate([np.arange(4096), np.arange(top - 4096, top),
                        rng.integers(0, top, 100000)]).astype(np.uint64)
    for khw in range(2, 65):
        mc = np.uint64(0xFFFFFFFF // khw + 1)
        # the quotient is first wrong just below a multiple of kH kW
        edge = k // np.uint64(khw) * np.uint64(khw) + np.uint64(khw - 1)
        for v in (k, edge[edge < top]):
            assert np.array_equal((v * mc) >> np.uint64(32), v // np.uint64(khw)), khw
    t = np.arange(64)
    for kw in range(1, 65):
        assert np.array_equal((t * (65535 // kw + 1)) >> 16, t // kw), kw


def test_three_bf16_parts_below_the_exact_range():
    """h + m + l holds every Float32 number of at least 2^-110, and is off by at
    most 2^-134 (half of the smallest bf16 denormal) below: the bound from which
    the kernels decide what to compute again (CPU model of the split)."""
    rng = np.random.default_rng(3)
    sig = 1.0 + rng.integers(0, 1 << 23, 4096) / float(1 << 23)
    for e in range(-149, -90):
        t = torch.from_numpy((sig * 2.0 ** e).astype(np.float32))
        h = t.bfloat16().float()
        m = (t - h).bfloat16().float()
        l = (t - h - m).bfloat16().float()
        off = (h.double() + m.double() + l.double() - t.double()).abs().max()
        assert float(off) <= (0.0 if e >= -110 else 2.0 ** -134), e


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(256, 292, 260), (1030, 1000, 257), (2049, 2000, 96),
                                   (4100, 4096, 64), (1, 4111, 4097), (16, 16, 2048)])
@pytest.mark.parametrize("side", ["row", "column"])
def test_small_elements_beside_large_ones(dev, M, N, K, side):
    """A row of A (a column of B) of ordinary and of tiny elements, where the
    ordinary ones meet zeros and the tiny ones large numbers: the outputs are
    sums of the tiny elements' products alone and as accurate as a Float32
    chain of K roundings (2-norm of the error 2^-24 sqrt(K) of the result);
    the outputs whose other operand is ordinary keep the split's accuracy."""
    g = torch.Generator(device="cuda").manual_seed(M + K)
    for e in (-112, -120, -126, -140):
        a = torch.randn((M, K), generator=g, device=dev)
        b = torch.randn((K, N), generator=g, device=dev)
        rows, cols = sorted({0, M // 2, M - 1}), sorted({0, N // 3, N - 1})
        if side == "row":
            a[rows, 1::2] *= 2.0 ** e
            b[:, cols] *= 2.0 ** 100
            b[::2, cols] = 0.0
        else:
            b[1::2, cols] *= 2.0 ** e
            a[rows, :] *= 2.0 ** 100
            a[rows, ::2] = 0.0
        got = mj.matmul(mj.Tensor(a), mj.Tensor(b)).torch.double()
        ref = a.double() @ b.double()
        mixed = torch.zeros((M, N), dtype=torch.bool, device=dev)
        mixed[np.ix_(rows, cols)] = True
        if side == "row":
            plain = ~mixed
            plain[:, cols] = False
        else:
            plain = ~mixed
            plain[rows, :] = False
        err = (got - ref)
        assert float(err[mixed].norm() / ref[mixed].norm()) <= 2.0 ** -24 * math.sqrt(K), e
        if bool(plain.any()):
            nk = -(-K // 32)
            assert float(err[plain].norm() / ref[plain].norm()) <= 2.0 ** -24 * math.sqrt(nk + 2), e


@pytest.mark.gpu
@pytest.mark.parametrize("n,c,h,w,oc", [(3, 40, 27, 31, 70), (16, 16, 60, 60, 128)])
def test_conv2d_small_elements_beside_large_ones(dev, n, c, h, w, oc):
    """The same for a convolution: one channel of ordinary numbers under zero
    weights, the others tiny under large weights."""
    g = torch.Generator(device="cuda").manual_seed(c)
    x = torch.randn((n, c, h, w), generator=g, device=dev)
    x[:, 1:] *= 2.0 ** -126
    conv = mj.Conv2d(c, oc, (3, 3), (1, 1), (1, 1))
    wt = torch.randn((oc, c, 3, 3), generator=g, device=dev) * 2.0 ** 100
    wt[:, 0] = 0.0
    conv.weight, conv.bias_t = mj.Tensor(wt), mj.Tensor(torch.zeros(oc, device=dev))
    got = conv.forward(mj.Tensor(x)).torch.cpu().double()
    ref = torch.nn.functional.conv2d(x.cpu().double(), wt.cpu().double(), padding=1)
    assert float((got - ref).norm() / ref.norm()) <= 2.0 ** -24 * math.sqrt(9 * c)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(4100, 4096, 70), (2049, 2000, 257), (1030, 1000, 96),
                                   (300, 517, 129), (33, 1000, 1030), (1, 4111, 4097),
                                   (16, 16, 2047)])
def test_whole_products_outside_the_split(dev, M, N, K):
    """Every output computed natively (all of A tiny), in every kernel and layout:
    one order of sums for all, at a Float32 chain's accuracy."""
    g = torch.Generator(device="cuda").manual_seed(K)
    a = torch.randn((M, K), generator=g, device=dev) * 2.0 ** -118
    b = torch.randn((K, N), generator=g, device=dev)
    ref, want = a.double() @ b.double(), None
    for la, lb in (("n", "t"), ("n", "n"), ("t", "n"), ("t", "t"), ("s", "n"), ("n", "s")):
        got = mj.matmul(mj.Tensor(_view(a, la)), mj.Tensor(_view(b, lb))).torch
        if want is None:
            assert float((got.double() - ref).norm() / ref.norm()) <= 2.0 ** -24 * math.sqrt(K)
            want = got
        assert torch.equal(got, want), (la, lb)


@pytest.mark.gpu
@pytest.mark.parametrize("n,c,h,w,oc", [(3, 40, 27, 31, 70), (16, 16, 60, 60, 128)])
def test_conv2d_outside_the_split_equals_matmul(dev, n, c, h, w, oc):
    """The same for a convolution (and infinities in some windows): the bits of
    the matmul on its im2col."""
    g = torch.Generator(device="cuda").manual_seed(oc)
    x = torch.randn((n, c, h, w), generator=g, device=dev) * 2.0 ** -118
    x[0, 1, 3, 4] = float("inf")
    conv = mj.Conv2d(c, oc, (3, 3), (1, 1), (1, 1))
    wt = torch.randn((oc, c, 3, 3), generator=g, device=dev)
    conv.weight, conv.bias_t = mj.Tensor(wt), mj.Tensor(torch.zeros(oc, device=dev))
    got = conv.forward(mj.Tensor(x)).torch
    cols = torch.nn.functional.unfold(x, (3, 3), padding=1)
    for i in range(n):
        want = mj.matmul(mj.Tensor(wt.reshape(oc, -1)), mj.Tensor(cols[i].contiguous())).torch
        np.testing.assert_array_equal(got[i].reshape(oc, -1).cpu().numpy(), want.cpu().numpy())


def _conv_against_matmul(dev, N, C, H, W, OC, kH, kW, s, pH, pW):
    """The convolution has the bits of the matmul on its im2col (torch's unfold:
    exact copies of the taps, zeros in the padding) plus the bias."""
    g = torch.Generator(device="cuda").manual_seed(C + kH * kW)
    x = torch.randn((N, C, H, W), generator=g, device=dev)
    conv = mj.Conv2d(C, OC, (kH, kW), (s, s), (pH, pW))
    wt = torch.randn((OC, C, kH, kW), generator=g, device=dev)
    b = torch.randn(OC, generator=g, device=dev)
    conv.weight, conv.bias_t = mj.Tensor(wt), mj.Tensor(b)
    got = conv.forward(mj.Tensor(x)).torch
    cols = torch.nn.functional.unfold(x, (kH, kW), padding=(pH, pW), stride=(s, s))
    wf = mj.Tensor(wt.reshape(OC, -1))
    for i in range(N):
        want = mj.matmul(wf, mj.Tensor(cols[i].contiguous())).torch + b[:, None]
        assert torch.equal(got[i].reshape(OC, -1), want), i


# N, C, H, W, OC, kH, kW, stride, pH, pW: more than 256^3 multiply-adds an image
CONV_MASK_SHAPES = [
    (8, 64, 80, 81, 70, 1, 1, 1, 0, 0),         # one tap a channel
    (32, 64, 56, 57, 64, 2, 2, 1, 1, 0),        # even kernel, padded on one side
    (9, 3, 150, 149, 64, 7, 7, 1, 3, 3),        # 49 taps: the mask's second word
    (4, 16, 70, 66, 64, 8, 8, 1, 4, 3),         # 64 taps
    (8, 8, 33, 150, 64, 1, 64, 1, 0, 31),       # a row of 64 taps
    (8, 8, 150, 33, 64, 64, 1, 1, 40, 0),       # a column of 64 taps
    (8, 8, 90, 95, 64, 2, 31, 1, 5, 40),        # padding wider than the kernel
    (32, 16, 100, 100, 16, 3, 3, 1, 1, 1),      # 16 channels out
]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", CONV_MASK_SHAPES)
def test_conv2d_masks_equal_matmul(dev, shape):
    _conv_against_matmul(dev, *shape)


CONV_ANY_SHAPES = [
    (8, 3, 128, 131, 64, 9, 9, 1, 4, 4),
    (16, 3, 227, 224, 64, 11, 11, 4, 2, 2),
    (2, 16, 60, 60, 128, 5, 13, 1, 2, 6),       # 65 taps
    (12, 24, 41, 37, 70, 11, 11, 1, 5, 5),
    (2, 8, 90, 90, 64, 3, 70, 1, 1, 35),        # wider than a mask word
    (32, 16, 56, 56, 128, 9, 9, 2, 4, 4),
]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", CONV_ANY_SHAPES)
def test_conv2d_more_than_64_taps_equals_matmul(dev, shape):
    _conv_against_matmul(dev, *shape)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N", [(4099, 4111), (70001, 257)])
def test_outer_products_are_correctly_rounded(dev, M, N):
    """K = 1: every output is the one product, rounded once."""
    g = torch.Generator(device="cuda").manual_seed(M)
    a, b = torch.randn((M, 1), generator=g, device=dev), torch.randn((1, N), generator=g, device=dev)
    for la, lb in (("n", "n"), ("n", "t"), ("t", "n")):
        assert torch.equal(mj.matmul(mj.Tensor(_view(a, la)), mj.Tensor(_view(b, lb))).torch, a * b)


@pytest.mark.gpu
@pytest.mark.parametrize("K", [2, 5, 15, 16, 17])
def test_short_sums_around_the_line(dev, K):
    """Both sides of the line at K = 16, all layouts, 128- and 64-row remainders:
    one order of sums for all layouts, and for K up to 16 as well for any number
    of rows and columns (one native chain); the error of at most K roundings."""
    M, N = 2900, 3001
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = torch.randn((M, K), generator=g, device=dev), torch.randn((K, N), generator=g, device=dev)
    ref, want = a.double() @ b.double(), None
    for la, lb in (("n", "t"), ("n", "n"), ("t", "n"), ("t", "t")):
        got = mj.matmul(mj.Tensor(_view(a, la)), mj.Tensor(_view(b, lb))).torch
        if want is None:
            assert float((got.double() - ref).norm() / ref.norm()) <= 2.0 ** -24 * math.sqrt(K)
            want = got
        assert torch.equal(got, want), (la, lb)
    few = mj.matmul(mj.Tensor(a[:100].contiguous()), mj.Tensor(b)).torch
    assert K > 16 or torch.equal(few, want[:100])


@pytest.mark.gpu
def test_dot_product_of_2_to_31_less_one(dev):
    """The last octet of k ends past 2^31 - 1: it holds the row's last elements
    and nothing beyond."""
    K = (1 << 31) - 1
    x, w = torch.zeros((1, K), device=dev), torch.zeros((K, 1), device=dev)
    for k, u, v in ((0, 1.5, 2.0), (1 << 30, -3.0, 0.25), (K - 8, 5.0, 3.0), (K - 1, 7.0, 4.0)):
        x[0, k], w[k, 0] = u, v
    assert float(mj.matmul(mj.Tensor(x), mj.Tensor(w)).torch) == 3.0 - 0.75 + 15.0 + 28.0


@pytest.mark.gpu
def test_row_strides_past_the_tiles_offsets(dev):
    """Rows 2^21 elements apart run the direct kernel: the bits of the product of
    the same rows side by side (as the left operand and as the right one)."""
    g = torch.Generator(device="cuda").manual_seed(21)
    M, N, K = 1000, 1030, 513                   # side by side: 64 x 64 tiles
    wide = torch.empty((M, 1 << 21), device=dev)
    a = wide[:, 5:5 + K]
    a.copy_(torch.randn((M, K), generator=g, device=dev))
    b = torch.randn((K, N), generator=g, device=dev)
    want = mj.matmul(mj.Tensor(a.contiguous()), mj.Tensor(b)).torch
    assert torch.equal(mj.matmul(mj.Tensor(a), mj.Tensor(b)).torch, want)
    want = mj.matmul(mj.Tensor(b.t()), mj.Tensor(a.contiguous().t())).torch
    assert torch.equal(mj.matmul(mj.Tensor(b.t()), mj.Tensor(a.t())).torch, want)


@pytest.mark.gpu
def test_rows_of_stride_zero(dev):
    """A row read by every output row (an expanded view)."""
    g = torch.Generator(device="cuda").manual_seed(22)
    a = torch.randn((1, 257), generator=g, device=dev)
    b = torch.randn((257, 1003), generator=g, device=dev)
    want = mj.matmul(mj.Tensor(a.expand(300, 257).contiguous()), mj.Tensor(b)).torch
    assert torch.equal(mj.matmul(mj.Tensor(a.expand(300, 257)), mj.Tensor(b)).torch, want)


@pytest.mark.gpu
def test_more_batches_than_a_grid_dimension(dev):
    """65537 products of K = 1030 in one call (two launches), against one by one."""
    g = torch.Generator(device="cuda").manual_seed(23)
    n, M, N, K = 65537, 2, 3, 1030
    a = torch.randn((n, M, K), generator=g, device=dev)
    b = torch.randn((n, K, N), generator=g, device=dev)
    got = mj.tensordot(mj.Tensor(a), mj.Tensor(b)).torch
    for i in (0, 1, 65534, 65535, 65536):
        assert torch.equal(got[i], mj.matmul(mj.Tensor(a[i]), mj.Tensor(b[i])).torch), i
    ref = (a.double().transpose(1, 2)[..., None] * b.double()[:, :, None, :]).sum(1)
    assert float((got.double() - ref).norm() / ref.norm()) <= 2.0 ** -24 * math.sqrt(K / 32 + 2)

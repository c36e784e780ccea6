"""Which kernel a call runs, as the library itself says (host only): the shapes
that the tests of each fp32 and bf16 kernel use reach it, so a change of a dispatch
rule that leaves a kernel without a test fails here."""
import pytest

import test_gpu_bf16_ring as ring
import test_gpu_conv2d as conv
import test_gpu_f32_split as split
import test_gpu_fp32 as fp32
from momijo_amd import _lib


def matmul(M, N, K, batches=1):
    return _lib.load().mj_matmul_f32_kernel(M, N, K, batches, K, 1).decode()


def conv2d(*shape):
    return _lib.load().mj_conv2d_f32_kernel(*shape).decode()


def bf16(M, N, K):
    return _lib.load().mj_gemm_bf16_kernel(M, N, K).decode()


def test_split_shapes_reach_every_split_kernel():
    took = {matmul(*s) for s in split._SHAPES}
    assert {"split 256x128", "split 128x128", "split 64x64", "split direct 32", "split direct 16",
            "split direct 16, 16 waves"} <= took


def test_the_split_tests_model_is_the_librarys_plan():
    for s in split._SHAPES:
        if s[2] > 16:
            name = matmul(*s).replace("split ", "").replace("direct ", "direct").replace(", 16 waves", "w16")
            assert split._plan(*s) == name, s


def test_native_shapes_reach_every_native_kernel():
    assert {matmul(*s) for s in fp32.NATIVE_SHAPES} == {
        "native 128x128", "native 64x64", "native tiny 32", "native tiny 16"}


def test_conv_shapes_reach_every_conv_kernel():
    assert {conv2d(*s) for s in conv._IM2COL_SHAPES + conv._NATIVE_SHAPES} >= {
        "native 32x32", "native 64x64", "native conv 224", "native conv 256", "split 64x64",
        "split 128x128"}
    def as_abi(n, c, h, w, oc, kh, kw, s, ph, pw):
        return n, c, h, w, oc, kh, kw, s, s, ph, pw
    assert {conv2d(*as_abi(*s)) for s in split.CONV_MASK_SHAPES} == {"split 64x64", "split 128x128"}
    assert {conv2d(*as_abi(*s)) for s in split.CONV_ANY_SHAPES} == {
        "split 64x64, any taps", "split 128x128, any taps"}


def test_bf16_shapes_reach_every_ring_tile():
    assert {bf16(*s) for s in ring._SHAPES} >= {"ring 32x32", "ring 64x64, 5 stages", "ring 64x64",
                                               "ring 128x64"}


@pytest.mark.parametrize("args,want", [
    ((256, 256, 256, 1, 256, 1), "native tiny 16"),      # 256^3 is the last native size
    ((257, 256, 256, 1, 256, 1), "split "),
    ((4096, 4096, 16, 1, 16, 1), "native 64x64"),        # K up to 16
    ((4096, 4096, 17, 1, 17, 1), "split 256x128"),
    ((1, 1, 1024, 1, 1024, 1), "native tiny 16"),        # K above 1024
    ((1, 1, 1025, 1, 1025, 1), "split direct 16, 16 waves"),
    ((512, 512, 1100, 1, (1 << 21) - 1, 1), "split direct"),
    ((4096, 4096, 64, 1, 1 << 21, 1), "split direct 32"),    # row strides past the tiles' offsets
    ((0, 5, 5, 1, 5, 1), ""),
])
def test_lines_of_the_rule(args, want):
    got = _lib.load().mj_matmul_f32_kernel(*args).decode()
    assert got.startswith(want) and (want or got == "")


def test_convolutions_past_the_tiles_offsets_run_direct():
    assert conv2d(1, 32, 4096, 4096, 32, 3, 3, 1, 1, 1, 1) == "split direct 32"

"""The 192 x 256 ring (tile configuration 13), forced: row counts around the
tile height, ragged columns, one K stage to many, whole tiles, K splits of
every tile and of a short last wave behind whole tiles, with and without bias,
and with the gated activation in its epilogue.  Bit-exact against the oracle; the activation bit-identical to
the GEMM followed by the activation kernel."""

import pytest
import torch

from helpers import announce
from minisgl_amd.kernel import act_and_mul_quant, gemm_act_supported, gemm_act_w8a8, gemm_w8a8
from minisgl_amd.kernel import lib as mw8lib
from test_gpu_gemm import _run_case

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CFG = 13


@pytest.fixture
def forced():
    lib = mw8lib.load()
    lib.mw8_set_tuning(-1, CFG, -1)
    assert lib.mw8_gemm_kernel_name(200, 512, 512) == b"tile3_gemm_kernel<192, 256, 128, 2, 4, 2>"
    yield lib
    lib.mw8_set_tuning(-1, -1, -1)


@pytest.mark.parametrize("M,N,K,bias", [
    (65, 256, 128, False), (191, 264, 256, True), (192, 256, 384, False), (193, 250, 512, True), (300, 1000, 640, False),
    (385, 513, 1024, True), (576, 768, 2048, False), (100, 4096, 4096, True), (3100, 4360, 256, False),
])
def test_forced(forced, M, N, K, bias):
    announce(f"192x256 M={M} N={N} K={K} bias={bias}")
    _run_case(M, K, N, seed=M + N + K, bias=bias)


# tail tiles, K ranges of each: behind one whole wave of 256 tiles, by row tiles
TAILS = [(300, 34816, 512, True, 16, 4), (100, 66000, 640, False, 2, 5), (3100, 4360, 768, True, 50, 5)]


@pytest.mark.parametrize("M,N,K,bias,tail,ranges", TAILS)
def test_split_last_wave(forced, M, N, K, bias, tail, ranges):
    announce(f"192x256 split last wave M={M} N={N} K={K} bias={bias}")
    assert -(-M // 192) * -(-N // 256) == 256 + tail
    assert forced.mw8_gemm_workspace_bytes(M, N, K) == tail * ranges * 192 * 256 * 4
    _run_case(M, K, N, seed=M + N, bias=bias)


@pytest.mark.parametrize("M,I,K,act,tail,ranges", [(300, 17408, 512, "silu", 16, 4), (3100, 2184, 768, "gelu", 50, 5)])
def test_activation_split_last_wave(forced, M, I, K, act, tail, ranges):
    assert -(-M // 192) * -(-2 * I // 256) == 256 + tail
    assert forced.mw8_gemm_act_workspace_bytes(M, I, K) == tail * ranges * 192 * 256 * 4
    test_activation(forced, M, I, K, act)


@pytest.mark.parametrize("M,I,K,act", [(192, 128, 128, "silu"), (200, 136, 512, "gelu"), (1000, 776, 1024, "silu"),
                                       (3100, 2184, 256, "silu")])
def test_activation(forced, M, I, K, act):
    announce(f"192x256 act M={M} I={I} K={K} {act}")
    gen = torch.Generator().manual_seed(M + I)
    q = torch.randint(-127, 128, (M, K), generator=gen, dtype=torch.int8).to(DEV)
    w = torch.randint(-127, 128, (2 * I, K), generator=gen, dtype=torch.int8).to(DEV)
    sa = (torch.rand(M, generator=gen) * 1e-3).to(DEV)
    sw = (torch.rand(2 * I, generator=gen) * 1e-2).to(DEV)
    assert gemm_act_supported(M, I, K)
    y = gemm_act_w8a8(q, sa, w, sw, act)
    forced.mw8_set_tuning(-1, 2, -1)
    want = act_and_mul_quant(gemm_w8a8(q, sa, w, sw), act, return_act=True)[2]
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))

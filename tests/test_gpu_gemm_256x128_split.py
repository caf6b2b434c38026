"""The 256 x 128 ring with its K split (tile configuration 3, forced): one
row tile and several, ragged rows and columns, the fewest
and the most K ranges, the grid just past the split, and the gated activation
in its reduction.  Bit-exact against the oracle; the activation bit-identical
to the GEMM followed by the activation kernel."""

import pytest
import torch

from helpers import announce
from minisgl_amd.kernel import act_and_mul_quant, gemm_act_supported, gemm_act_w8a8, gemm_w8a8
from minisgl_amd.kernel import lib as mw8lib
from test_gpu_gemm import _run_case

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CFG, TILE = 3, 256 * 128 * 4


@pytest.fixture
def forced():
    lib = mw8lib.load()
    lib.mw8_set_tuning(-1, CFG, -1)
    yield lib
    lib.mw8_set_tuning(-1, -1, -1)


# K ranges: four K stages or 16 ranges or 256 / tiles, whichever is fewest; none below four
@pytest.mark.parametrize("M,N,K,bias,parts", [
    (130, 1000, 2048, True, 8 * 16), (256, 128, 512, False, 4), (255, 513, 384, False, 0), (257, 250, 1152, True, 4 * 9),
    (600, 1928, 640, False, 48 * 5), (1000, 2048, 1024, True, 64 * 4), (1030, 1664, 1024, False, 0),
])
def test_forced(forced, M, N, K, bias, parts):
    announce(f"256x128 split M={M} N={N} K={K} bias={bias}")
    assert forced.mw8_gemm_workspace_bytes(M, N, K) == parts * TILE
    _run_case(M, K, N, seed=M + N + K, bias=bias)


@pytest.mark.parametrize("M,I,K,act", [(200, 136, 512, "gelu"), (1030, 776, 1024, "silu"), (256, 64, 4096, "silu")])
def test_activation(forced, M, I, K, act):
    announce(f"256x128 split act M={M} I={I} K={K} {act}")
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


def test_picked():
    """The automatic choice: a decode batch past 128 rows through a deep K."""
    assert mw8lib.load().mw8_gemm_kernel_name(256, 5120, 17408) == b"tile3_gemm_kernel<256, 128, 128, 4, 2, 3>"
    _run_case(131, 8704, 4096, seed=1)

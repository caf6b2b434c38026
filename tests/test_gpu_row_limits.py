"""As many long rows as fit the card: the blocks stay small enough for a
launch's 2^32 threads.  In place, so that one buffer of 180 GB is all; a
sample of rows is compared with the oracle."""

import pytest
import torch

from helpers import announce, bf16_bits_equal, f32
from minisgl_amd.kernel import rmsnorm_quant
from oracle import w8a8 as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("H", [10760])
def test_norm_of_many_long_rows(H):
    M = 1 << 23  # blocks of 512 threads would be 2^32 threads
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 2 * M * H + (8 << 30):
        pytest.skip("needs 188 GB of free device memory")
    announce(f"norm rows {M} x {H} in place")
    gen = torch.Generator().manual_seed(H)
    rows = torch.tensor([0, 1, M // 2 - 1, M // 2, M - 2, M - 1])
    x = torch.randn(len(rows), H, generator=gen).to(torch.bfloat16)
    w = (torch.rand(H, generator=gen) + 0.5).to(torch.bfloat16)
    xd = torch.empty((M, H), dtype=torch.bfloat16, device=DEV)
    xd[rows.to(DEV)] = x.to(DEV)
    rmsnorm_quant(xd, w.to(DEV), 1e-6, y=xd, quantize=False)
    got = xd[rows.to(DEV)]
    del xd
    torch.cuda.empty_cache()
    assert bf16_bits_equal(got, orc.rmsnorm_quant(f32(x), f32(w), 1e-6)[2]).all()

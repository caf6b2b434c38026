"""Rows of more than 8192 elements at the edges of the 2 - 9 vectors a thread
holds, and at row counts around the blocks that are resident at once (512 -
2560 rows).  Bit-exact against the oracle (the activation: its requant
against the oracle on the kernel's own activation)."""

import numpy as np
import pytest
import torch

from helpers import announce, bf16_bits_equal, f32
from minisgl_amd.kernel import act_and_mul_quant, quant_per_token, rmsnorm_quant
from oracle import w8a8 as orc
from test_gpu_row_shapes import DEV, _rows, _x

pytestmark = pytest.mark.gpu

EDGES = [1536, 1537, 2560, 2561, 3584, 3585, 4096]  # vectors of 8 elements
# (rows, vectors): 4 - 9 vectors per thread with every block resident, and the row past it
RESIDENT = [(600, 1300), (768, 2176), (769, 2176), (1024, 2560), (1025, 2560), (1280, 2560), (1281, 2560), (2048, 2300),
            (2049, 2300)]


def _check_quant(q, s, r, x):
    q_ref, s_ref = orc.quant_per_token(x)
    np.testing.assert_array_equal(q.cpu().numpy()[r], q_ref)
    np.testing.assert_array_equal(s.cpu().numpy()[r].view(np.uint32), s_ref.view(np.uint32))


@pytest.mark.parametrize("M,nvec", [(514, n) for n in EDGES] + RESIDENT)
def test_quant_long_rows(M, nvec):
    announce(f"quant long rows {M} x {8 * nvec}")
    x = _x(M, 8 * nvec, nvec)
    q, s = quant_per_token(x.to(DEV))
    r = _rows(M)
    _check_quant(q, s, r, f32(x[r]))


@pytest.mark.parametrize("M,nvec", [(514, n) for n in EDGES] + RESIDENT)
def test_act_long_rows(M, nvec):
    announce(f"act long rows {M} x {8 * nvec}")
    x = _x(M, 16 * nvec, nvec)
    q, s, a = act_and_mul_quant(x.to(DEV), "silu" if nvec % 2 else "gelu", return_act=True)
    r = _rows(M)
    want = (orc.silu_and_mul if nvec % 2 else orc.gelu_and_mul)(f32(x[r]))
    got = f32(a[torch.as_tensor(r, device=DEV)])
    assert np.linalg.norm(got - want) <= 1e-3 * np.linalg.norm(want)
    _check_quant(q, s, r, got)


@pytest.mark.parametrize("M,nvec", [(514, n) for n in EDGES] + RESIDENT)
def test_norm_long_rows(M, nvec):
    announce(f"norm long rows {M} x {8 * nvec}")
    H = 8 * nvec
    x, res = _x(M, H, M), _x(M, H, nvec)
    w = (torch.rand(H, generator=torch.Generator().manual_seed(3)) + 0.5).to(torch.bfloat16)
    r = _rows(M)
    rdev = torch.as_tensor(r, device=DEV)
    rd = res.to(DEV)
    q, s, y = rmsnorm_quant(x.to(DEV), w.to(DEV), 1e-6, residual=rd, return_y=True)
    q_ref, s_ref, y_ref, h_ref = orc.rmsnorm_quant(f32(x[r]), f32(w), 1e-6, residual=f32(res[r]))
    assert bf16_bits_equal(rd[rdev], h_ref).all() and bf16_bits_equal(y[rdev], y_ref).all()
    np.testing.assert_array_equal(q.cpu().numpy()[r], q_ref)
    np.testing.assert_array_equal(s.cpu().numpy()[r].view(np.uint32), s_ref.view(np.uint32))
    plain = rmsnorm_quant(x.to(DEV), w.to(DEV), 1e-6, quantize=False)
    assert bf16_bits_equal(plain[rdev], orc.rmsnorm_quant(f32(x[r]), f32(w), 1e-6)[2]).all()

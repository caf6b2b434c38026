"""The row kernels (quantizer, activation + requant, RMSNorm) at the edges
of their thread layouts: row lengths around 16, 32, 64, 96, 512, 1024 and
4096 vectors of 8, and row counts around the choices that depend on them.
Bit-exact against the oracle (the activation: its requant against the
oracle on the kernel's own activation, row by row)."""

import numpy as np
import pytest
import torch

from helpers import announce, bf16_bits_equal, f32
from minisgl_amd.kernel import act_and_mul_quant, quant_per_token, rmsnorm_quant, rmsnorm_strided
from oracle import w8a8 as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# (rows, vectors of 8 elements)
SHAPES = [(5, 1), (17, 15), (33, 16), (9, 17), (7, 32), (6, 33), (5, 64), (5, 65), (3, 96), (3, 97), (8193, 64),
          (5462, 96), (5500, 96), (5000, 128), (1100, 512), (1024, 512), (800, 513), (1023, 513), (4096, 513),
          (4097, 769), (700, 1024), (512, 1025), (513, 1025), (2, 3072), (3, 4096), (514, 1100)]


def _x(M, K, seed):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=gen)
    x[torch.rand(M, K, generator=gen) < 1e-3] *= 20
    x[M // 2] = 0
    return x.to(torch.bfloat16)


def _rows(M):
    return np.unique(np.r_[0, 1 % M, M // 2, M - 1, np.random.default_rng(M).integers(0, M, 40)])


@pytest.mark.parametrize("M,nvec", SHAPES)
def test_quant_rows(M, nvec):
    announce(f"quant rows {M} x {8 * nvec}")
    x = _x(M, 8 * nvec, M + nvec)
    q, s = quant_per_token(x.to(DEV))
    r = _rows(M)
    q_ref, s_ref = orc.quant_per_token(f32(x[r]))
    np.testing.assert_array_equal(q.cpu().numpy()[r], q_ref)
    np.testing.assert_array_equal(s.cpu().numpy()[r].view(np.uint32), s_ref.view(np.uint32))


@pytest.mark.parametrize("M,nvec", [s for s in SHAPES if s[0] * s[1] < 2_000_000])
def test_act_rows(M, nvec):
    announce(f"act rows {M} x {8 * nvec}")
    x = _x(M, 16 * nvec, M + nvec)
    q, s, a = act_and_mul_quant(x.to(DEV), "silu" if nvec % 2 else "gelu", return_act=True)
    r = _rows(M)
    d = 8 * nvec
    want = (orc.silu_and_mul if nvec % 2 else orc.gelu_and_mul)(f32(x[r]))
    got = f32(a[torch.as_tensor(r, device=DEV)])
    assert got.shape == (len(r), d) and np.linalg.norm(got - want) <= 1e-3 * np.linalg.norm(want)
    q_ref, s_ref = orc.quant_per_token(got)
    np.testing.assert_array_equal(q.cpu().numpy()[r], q_ref)
    np.testing.assert_array_equal(s.cpu().numpy()[r].view(np.uint32), s_ref.view(np.uint32))


@pytest.mark.parametrize("M,nvec", SHAPES)
def test_norm_rows(M, nvec):
    announce(f"norm rows {M} x {8 * nvec}")
    H = 8 * nvec
    x, res = _x(M, H, M), _x(M, H, nvec)
    w = (torch.rand(H, generator=torch.Generator().manual_seed(3)) + 0.5).to(torch.bfloat16)
    r = _rows(M)
    rd = res.to(DEV)
    q, s, y = rmsnorm_quant(x.to(DEV), w.to(DEV), 1e-6, residual=rd, return_y=True)
    q_ref, s_ref, y_ref, h_ref = orc.rmsnorm_quant(f32(x[r]), f32(w), 1e-6, residual=f32(res[r]))
    rdev = torch.as_tensor(r, device=DEV)
    assert bf16_bits_equal(rd[rdev], h_ref).all() and bf16_bits_equal(y[rdev], y_ref).all()
    np.testing.assert_array_equal(q.cpu().numpy()[r], q_ref)
    np.testing.assert_array_equal(s.cpu().numpy()[r].view(np.uint32), s_ref.view(np.uint32))


@pytest.mark.parametrize("G,heads,D", [(1, 1, 8), (3, 5, 64), (2080, 9, 128), (777, 3, 256), (70, 7, 136)])
def test_head_norm_in_place(G, heads, D):
    announce(f"head norm {G} x {heads} x {D}")
    width = (heads + 2) * D
    x = _x(G, width, G + D)
    w = (torch.rand(D, generator=torch.Generator().manual_seed(4)) + 0.5).to(torch.bfloat16)
    xd = x.to(DEV)
    assert rmsnorm_strided(xd[:, : heads * D].view(G, heads, D), w.to(DEV), 1e-6)
    want = orc.rmsnorm_quant(f32(x[:, : heads * D]).reshape(-1, D), f32(w), 1e-6)[2]
    assert bf16_bits_equal(xd[:, : heads * D].reshape(-1, D), want).all()
    assert torch.equal(xd[:, heads * D :].cpu().view(torch.int16), x[:, heads * D :].view(torch.int16))

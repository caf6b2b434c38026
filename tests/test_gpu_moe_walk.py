"""The grouped walk (moe cfg 2) where it can go wrong: chunk heights around
the 16-row fragments, the 128-row DMA variant and the 192-row chunk limit,
empty experts, the fewest K stages, more items than blocks (the ring runs on
across items), and the fused activation.  Bit-exact against the oracle's
grouped GEMM; the fused activation bit-identical to the GEMM followed by the
activation kernel."""

import numpy as np
import pytest
import torch

from helpers import announce, bf16_bits_equal
from minisgl_amd.kernel import (
    act_and_mul_quant,
    fused_moe_kernel_act_w8a8,
    fused_moe_kernel_w8a8,
    moe_align_block_size,
    moe_gemm_act_preferred,
    quant_per_token,
)
from minisgl_amd.kernel import lib as mw8lib
from oracle import w8a8 as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# pairs per expert: fragment, DMA-variant and chunk edges, none, several chunks
COUNTS = [1, 15, 16, 17, 0, 64, 65, 127, 128, 129, 175, 191, 192, 193, 0, 256, 257, 320, 383, 384, 385, 31, 33, 0]


def _case(counts, k, N, K, seed):
    """Hand-made routing: pair p of the flat [M, k] ids goes to the expert
    that a shuffled list of the counts gives it."""
    gen = torch.Generator().manual_seed(seed)
    flat = torch.cat([torch.full((c,), e, dtype=torch.int32) for e, c in enumerate(counts)])
    flat = flat[torch.randperm(flat.numel(), generator=gen)]
    pad = -flat.numel() % k
    flat = torch.cat([flat, flat[:pad]])
    ids = flat.view(-1, k).contiguous()
    E = len(counts)
    W = torch.randint(-127, 128, (E, N, K), generator=gen, dtype=torch.int8)
    SW = torch.rand(E, N, generator=gen) * 1e-2 + 1e-4
    tw = torch.rand(ids.shape, generator=gen)
    return ids, W, SW, tw, gen


@pytest.mark.parametrize("B", [64, 128])
@pytest.mark.parametrize("N,K", [(256, 640), (4096, 640), (512, 1152)])
def test_walk_equals_oracle(N, K, B):
    k = 2
    ids, W, SW, tw, gen = _case(COUNTS, k, N, K, N + K)
    M, E = ids.shape[0], W.shape[0]
    idsd, twd, Wd, SWd = ids.to(DEV), tw.to(DEV), W.to(DEV), SW.to(DEV)
    sorted_ids, expert_ids, npp = moe_align_block_size(idsd, B, E)
    lib = mw8lib.load()
    try:
        lib.mw8_set_tuning(-1, -1, 2)
        for which in (1, 2):
            announce(f"walk N={N} K={K} B={B} gemm{which}")
            rows = M if which == 1 else M * k
            q, s = quant_per_token(torch.randn(rows, K, generator=gen).to(torch.bfloat16).to(DEV))
            top_k, routed = (k, None) if which == 1 else (1, tw.numpy())
            y_ref = orc.grouped_gemm_w8a8(q.cpu().numpy(), s.cpu().numpy(), W.numpy(), SW.numpy(), ids.numpy(), top_k,
                                          routed=routed)
            out = torch.empty(M * k, N, dtype=torch.bfloat16, device=DEV)
            for _ in range(2):
                out.zero_()
                fused_moe_kernel_w8a8(q, s, Wd, SWd, out, twd, sorted_ids, expert_ids, npp, routed is not None, top_k,
                                      B, M * k)
                torch.cuda.synchronize()
                assert bf16_bits_equal(out, y_ref).all()
    finally:
        lib.mw8_set_tuning(-1, -1, -1)


@pytest.mark.parametrize("act", ["silu", "gelu"])
@pytest.mark.parametrize("routed", [False, True])
def test_walk_activation_equals_separate(act, routed):
    k, N, K, B = 2, 2048, 768, 64
    ids, W, SW, tw, gen = _case(COUNTS, k, N, K, 11)
    M, E = ids.shape[0], W.shape[0]
    idsd, twd, Wd, SWd = ids.to(DEV), tw.to(DEV), W.to(DEV), (SW * 1e-2).to(DEV)
    assert moe_gemm_act_preferred(M * k, N, K, E)
    sorted_ids, expert_ids, npp = moe_align_block_size(idsd, B, E)
    q, s = quant_per_token(torch.randn(M, K, generator=gen).to(torch.bfloat16).to(DEV))
    announce(f"walk activation {act} routed={routed}")
    lib = mw8lib.load()
    try:
        lib.mw8_set_tuning(-1, -1, 0)  # one tile per alignment block
        c1 = torch.empty(M * k, N, dtype=torch.bfloat16, device=DEV)
        fused_moe_kernel_w8a8(q, s, Wd, SWd, c1, twd, sorted_ids, expert_ids, npp, routed, k, B, M * k)
        lib.mw8_set_tuning(-1, -1, 2)
        out = torch.empty(M * k, N // 2, dtype=torch.bfloat16, device=DEV)
        fused_moe_kernel_act_w8a8(q, s, Wd, SWd, out, sorted_ids, expert_ids, npp, k, B, M * k, act,
                                  twd if routed else None)
        torch.cuda.synchronize()
    finally:
        lib.mw8_set_tuning(-1, -1, -1)
    want = act_and_mul_quant(c1, act, return_act=True)[2]
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))


def _any_order(sorted_ids, expert_ids, npp, B, E, numel, seed):
    """The same pairs in lists that the alignment would not write: blocks in
    random order, padding between the pairs of a block, blocks of experts
    outside [0, E) that name real pairs, a last block in use only in part and
    room behind it."""
    gen = torch.Generator().manual_seed(seed)
    nb = int(npp.item()) // B
    blocks, experts = sorted_ids[: nb * B].view(nb, B).cpu(), expert_ids[:nb].cpu()
    few = (blocks < numel).sum(1).argmin()
    last, last_e = blocks[few : few + 1], experts[few : few + 1]
    keep = torch.arange(nb) != few
    blocks, experts = blocks[keep], experts[keep]
    blocks = blocks.gather(1, torch.rand(blocks.shape, generator=gen).argsort(1))
    foreign = torch.arange(4 * B, dtype=torch.int32).view(4, B) % numel
    blocks = torch.cat([blocks, foreign])
    experts = torch.cat([experts, torch.tensor([-1, E, E + 7, -5], dtype=torch.int32)])
    order = torch.randperm(len(experts), generator=gen)
    blocks = torch.cat([blocks[order], last, torch.zeros(2, B, dtype=torch.int32)])
    experts = torch.cat([experts[order], last_e, torch.zeros(2, dtype=torch.int32)])
    used = (len(experts) - 3) * B + int((last < numel).sum())
    return blocks.reshape(-1).to(DEV), experts.to(DEV), torch.tensor([used], dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("B", [64, 128])
@pytest.mark.parametrize("few_pairs", [False, True])
def test_lists_in_any_order(B, few_pairs):
    """Lists whose blocks are not sorted by expert, in every configuration:
    the grouped GEMM takes the expert of each alignment block from
    expert_ids, whatever its neighbours are."""
    k, N, K = 2, 512, 640
    counts = [3, 0, 17, 2, 30, 1, 9, 0, 40, 5] if few_pairs else COUNTS
    ids, W, SW, tw, gen = _case(counts, k, N, K, 21 + B)
    M, E = ids.shape[0], W.shape[0]
    idsd, twd, Wd, SWd = ids.to(DEV), tw.to(DEV), W.to(DEV), (SW * 1e-2).to(DEV)
    aligned = moe_align_block_size(idsd, B, E)
    lists = _any_order(*aligned, B, E, M * k, B)
    q, s = quant_per_token(torch.randn(M, K, generator=gen).to(torch.bfloat16).to(DEV))
    y_ref = orc.grouped_gemm_w8a8(q.cpu().numpy(), s.cpu().numpy(), W.numpy(), SWd.cpu().numpy(), ids.numpy(), k,
                                  routed=tw.numpy())
    lib = mw8lib.load()
    try:
        for cfg in (0, -1, 1, 2):
            announce(f"any order B={B} few={few_pairs} cfg {cfg}")
            lib.mw8_set_tuning(-1, -1, cfg)
            out = torch.zeros(M * k, N, dtype=torch.bfloat16, device=DEV)
            fused_moe_kernel_w8a8(q, s, Wd, SWd, out, twd, *lists, True, k, B, M * k)
            torch.cuda.synchronize()
            assert bf16_bits_equal(out, y_ref).all()
        want = act_and_mul_quant(out, "silu", return_act=True)[2]
        for cfg in (-1, 1, 2):
            announce(f"any order B={B} few={few_pairs} activation cfg {cfg}")
            lib.mw8_set_tuning(-1, -1, cfg)
            act = torch.zeros(M * k, N // 2, dtype=torch.bfloat16, device=DEV)
            fused_moe_kernel_act_w8a8(q, s, Wd, SWd, act, *lists, k, B, M * k, "silu", twd)
            torch.cuda.synchronize()
            assert torch.equal(act.view(torch.int16), want.view(torch.int16))
    finally:
        lib.mw8_set_tuning(-1, -1, -1)


@pytest.mark.parametrize("used", [0, -64])
def test_no_blocks_in_use(used):
    """Nothing is written where num_post_pad says that no block is in use."""
    ids, W, SW, tw, gen = _case([5, 3], 2, 256, 640, 4)
    M, E = ids.shape[0], W.shape[0]
    sorted_ids, expert_ids, npp = moe_align_block_size(ids.to(DEV), 64, E)
    npp.fill_(used)
    q, s = quant_per_token(torch.randn(M, 640, generator=gen).to(torch.bfloat16).to(DEV))
    lib = mw8lib.load()
    try:
        for cfg in (0, 1, 2):
            announce(f"no blocks in use: {used}, cfg {cfg}")
            lib.mw8_set_tuning(-1, -1, cfg)
            out = torch.full((M * 2, 256), 7, dtype=torch.bfloat16, device=DEV)
            fused_moe_kernel_w8a8(q, s, W.to(DEV), SW.to(DEV), out, tw.to(DEV), sorted_ids, expert_ids, npp, False, 2,
                                  64, M * 2)
            torch.cuda.synchronize()
            assert (out == 7).all()
    finally:
        lib.mw8_set_tuning(-1, -1, -1)


def test_walk_preference_is_host_only():
    assert moe_gemm_act_preferred(2400, 1536, 2048, 128)
    assert not moe_gemm_act_preferred(100, 1536, 512, 128)  # four K stages: below the walk's fewest
    assert moe_gemm_act_preferred(32 * 128, 1536, 512, 128)
    assert not moe_gemm_act_preferred(2400, 1536, 2040, 128)


@pytest.mark.parametrize("tokens,top_k,E,H,I", [(12, 4, 8, 1024, 768), (40, 2, 32, 1024, 1408), (130, 2, 16, 1024, 1408),
                                                (700, 2, 8, 1024, 768), (4000, 2, 8, 256, 640)])
def test_layer_equals_forced_tiles(tokens, top_k, E, H, I):
    """A layer on each side of the choice between the tiles, the chunk walk
    and the tall walk: the bits of the tiles."""
    from minisgl_amd.moe.fused import fused_experts_impl_w8a8

    announce(f"walk choice T={tokens} k={top_k} E={E} H={H} I={I}")
    gen = torch.Generator().manual_seed(tokens + E)
    w1 = torch.randint(-127, 128, (E, 2 * I, H), generator=gen, dtype=torch.int8).to(DEV)
    w2 = torch.randint(-127, 128, (E, H, I), generator=gen, dtype=torch.int8).to(DEV)
    s1, s2 = (torch.rand(E, n, generator=gen).to(DEV) * 1e-3 for n in (2 * I, H))
    x = torch.randn(tokens, H, generator=gen).to(torch.bfloat16).to(DEV)
    ids = torch.rand(tokens, E, generator=gen).topk(top_k, dim=1).indices.int().to(DEV)
    tw = torch.rand(tokens, top_k, generator=gen).to(DEV)
    lib = mw8lib.load()
    got = fused_experts_impl_w8a8(x.clone(), w1, s1, w2, s2, tw, ids)
    try:
        lib.mw8_set_tuning(-1, -1, 0)
        want = fused_experts_impl_w8a8(x.clone(), w1, s1, w2, s2, tw, ids)
    finally:
        lib.mw8_set_tuning(-1, -1, -1)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))

"""Batched experts on the matrix cores with fp32 hidden states, and batches
whose experts hold many pairs, against float64."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from fastkernels_amd.kernels import hip

pytestmark = pytest.mark.gpu


def _randn(gen, shape, scale=1.0, dtype=torch.bfloat16):
    return (torch.randn(shape, generator=gen) * scale).to(dtype).cuda()


def _mlp(x, gu, dn):
    g, u = (x @ gu.double().t()).chunk(2, dim=-1)
    return (F.silu(g) * u) @ dn.double().t()


def _reference(x, ids, w, gu, dn, sgu=None, sdn=None, sg=None):
    xd = x.double()
    out = torch.zeros_like(xd)
    for e in range(gu.shape[0]):
        share = (w.double() * (ids == e)).sum(-1, keepdim=True)
        t = (share != 0).nonzero()[:, 0]
        if len(t):
            out[t] += share[t] * _mlp(xd[t], gu[e], dn[e])
    if sgu is not None:
        s = _mlp(xd, sgu, sdn)
        out += s if sg is None else torch.sigmoid(xd @ sg.double().reshape(-1, 1)) * s
    return out


# tiles of 16 and 32 pairs (the average pairs per expert either side of the
# line), one pair, a tile's edge, several tiles of one expert; with and
# without the shared expert; the shapes the kernels take
@pytest.mark.parametrize("tokens,hidden,inter,experts,top_k,shared", [
    (84, 2048, 512, 256, 8, True),
    (96, 512, 256, 16, 2, True),     # 12 pairs on average: tiles of 16
    (97, 512, 256, 16, 2, False),    # just over: tiles of 32
    (150, 1024, 256, 4, 3, True),    # 112 pairs an expert: further tiles
    (300, 1024, 512, 3, 2, False),
    (512, 2048, 256, 256, 8, True),
    # routed experts alone: fewer pairs than the fp32 line (3 an expert of 2048 x 512) and at it
    (95, 2048, 512, 64, 2, False),
    (96, 2048, 512, 64, 2, False),
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_expert_batches(tokens, hidden, inter, experts, top_k, shared, dtype):
    gen = torch.Generator().manual_seed(tokens)
    gu, dn = _randn(gen, (experts, 2 * inter, hidden), 0.02), _randn(gen, (experts, hidden, inter), 0.02)
    x = _randn(gen, (tokens, hidden), 1.0, dtype)
    ids = torch.rand((tokens, experts), generator=gen).topk(top_k, dim=-1).indices
    ids[:17] = ids[0]  # one set of experts with more pairs than the others
    ids, w = ids.to(torch.int32).cuda(), torch.rand((tokens, top_k), generator=gen).cuda()
    if shared:
        s = (_randn(gen, (2 * inter, hidden), 0.02), _randn(gen, (hidden, inter), 0.02), _randn(gen, (hidden,), 0.02))
        out = hip.hip_qwen36_batched_routed_shared_experts_decode(x, ids, w, gu, dn, *s)
    else:
        s = ()
        out = hip.hip_qwen36_batched_routed_experts_decode(x, ids, w, gu, dn)
    ref = _reference(x, ids, w, gu, dn, *s)
    # fp32: sums over K = H then I with about K / 100 roundings of 2^-24; bf16
    # hidden states: the activations as two bf16 terms, 2^-18 of each rounded
    err = float((out.double() - ref).norm() / ref.norm())
    assert err < (1e-6 if dtype == torch.float32 else 8e-6), err
    again = (hip.hip_qwen36_batched_routed_shared_experts_decode(x, ids, w, gu, dn, *s) if shared
             else hip.hip_qwen36_batched_routed_experts_decode(x, ids, w, gu, dn))
    assert torch.equal(out, again)


def test_one_expert_takes_every_pair():
    gen = torch.Generator().manual_seed(9)
    gu, dn = _randn(gen, (8, 512, 512), 0.02), _randn(gen, (8, 512, 256), 0.02)
    x = _randn(gen, (200, 512), 1.0, torch.float32)
    ids, w = torch.full((200, 2), 5, dtype=torch.int64).cuda(), torch.rand((200, 2), generator=gen).cuda()
    out = hip.hip_qwen36_batched_routed_experts_decode(x, ids, w, gu, dn)
    ref = _reference(x, ids, w, gu, dn)
    assert float((out.double() - ref).norm() / ref.norm()) < 1e-6


def test_values_past_the_bf16_range():
    """fp32 hidden states above the largest bf16 (3.39e38), against weights that bring them back into range."""

    gen = torch.Generator().manual_seed(11)
    gu, dn = _randn(gen, (8, 512, 512), 0.02), _randn(gen, (8, 512, 256), 0.02)
    x = _randn(gen, (100, 512), 1.0, torch.float32)
    x[::7, 9] = 3.4e38
    gu[:, :, 9] = 1e-38
    ids = torch.rand((100, 8), generator=gen).topk(2, dim=-1).indices.cuda()
    w = torch.rand((100, 2), generator=gen).cuda()
    out = hip.hip_qwen36_batched_routed_experts_decode(x, ids, w, gu, dn)
    ref = _reference(x, ids, w, gu, dn)
    assert float((out.double() - ref).norm() / ref.norm()) < 1e-6


@pytest.mark.parametrize("pairs,experts", [(1, 1), (63, 3), (64, 256), (65, 2), (128, 256), (136, 1000), (40, 8), (1023, 7), (1030, 1024), (4096, 256), (4096, 1)])
def test_routing_tables(pairs, experts):
    from oracle import qwen36 as oracle

    gen = torch.Generator().manual_seed(pairs)
    top_k = 8 if pairs % 8 == 0 else 1  # (a token may name an expert twice here)
    ids = torch.randint(0, experts, (pairs // top_k, top_k), generator=gen)
    got = hip.hip_qwen36_moe_align(ids.cuda(), experts)
    for g, r in zip(got, oracle.moe_align(ids, experts)):
        assert torch.equal(g.cpu(), torch.from_numpy(r))


# past the tagged router's 256 tokens: logits as tiles, then the selection
@pytest.mark.parametrize("tokens,hidden,experts,top_k,bias,dtype", [
    (257, 2048, 256, 8, False, torch.float32),
    (300, 512, 48, 3, True, torch.bfloat16),
    (512, 1024, 1024, 8, True, torch.float32),
    (20, 64, 272, 8, False, torch.float32),
    # more than 256 experts or 2,048 values: either side of the line between the kernels
    (1, 512, 1024, 8, True, torch.float32),
    (4, 512, 1024, 8, False, torch.bfloat16),
    (5, 512, 1024, 8, False, torch.bfloat16),
    (64, 4096, 256, 8, False, torch.float32),
    (65, 4096, 256, 8, True, torch.float32),
    (112, 3072, 16, 4, True, torch.float32),
])
def test_router_batches(tokens, hidden, experts, top_k, bias, dtype):
    from oracle import qwen36 as oracle

    gen = torch.Generator().manual_seed(tokens)
    x, norm = _randn(gen, (tokens, hidden), 1.0, dtype), _randn(gen, (hidden,), 0.1)
    w = _randn(gen, (experts, hidden), 0.05)
    b = _randn(gen, (experts,), 0.5, torch.float32) if bias else None
    logits, ids, weights = hip.hip_qwen36_batched_moe_router_decode(x, norm, w, top_k=top_k, router_bias=b)
    ref, _, _ = oracle.router(x.cpu(), norm.cpu(), w.cpu(), top_k, router_bias=None if b is None else b.cpu(), dtype=torch.float64)
    # 2^-24 of sum |w| |x| per rounding of the K / 64 partial sums
    bound = (hidden / 64 + 20) * 2.0 ** -24 * hidden ** 0.5 * 0.05 * hidden ** 0.5
    assert float((logits.cpu().double() - ref).abs().max()) < bound
    own = torch.softmax(logits.cpu().double(), -1)
    val, own_ids = oracle.topk_lowest_id(torch.softmax(logits.cpu(), -1), top_k)
    assert torch.equal(ids.cpu(), own_ids)
    pick = own.gather(1, own_ids)
    assert torch.allclose(weights.cpu().double(), pick / pick.sum(-1, keepdim=True), rtol=1e-5, atol=0)

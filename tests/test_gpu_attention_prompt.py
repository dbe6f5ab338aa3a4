"""Attention over many rows of one sequence in one call, against the oracle's
maths in float64 and against calls of a few rows."""

from __future__ import annotations

import pytest
import torch

from fastkernels_amd import _lib
from fastkernels_amd.kernels import hip
from fastkernels_amd.plan import AttentionStepPlan

pytestmark = pytest.mark.gpu


def _randn(gen, shape, scale=1.0, dtype=torch.bfloat16):
    return (torch.randn(shape, generator=gen) * scale).to(dtype).cuda()


def _inputs(seed, tokens, hidden, heads, kvh, positions, x_dtype, cache_dtype):
    gen = torch.Generator().manual_seed(seed)
    w = dict(
        norm_weight=_randn(gen, (hidden,), 0.1), q_proj_weight=_randn(gen, (2 * heads * 256, hidden), 0.02),
        k_proj_weight=_randn(gen, (kvh * 256, hidden), 0.02), v_proj_weight=_randn(gen, (kvh * 256, hidden), 0.02),
        out_proj_weight=_randn(gen, (hidden, heads * 256), 0.02), q_norm_weight=_randn(gen, (256,), 0.1),
        k_norm_weight=_randn(gen, (256,), 0.1))
    x = _randn(gen, (tokens, hidden), 1.0, x_dtype)
    kc, vc = (_randn(gen, (positions, kvh, 256), 1.0, cache_dtype) for _ in range(2))
    return x, kc, vc, w


def _reference(x, kc, vc, w, start, heads, kvh, rope_dim, theta, interleaved):
    d = {k: v.double() for k, v in w.items()}
    norm = lambda v, g: v * torch.rsqrt((v * v).mean(-1, keepdim=True) + 1e-6) * (1.0 + g)  # noqa: E731
    tokens, xd = x.shape[0], x.double()
    xn = norm(xd, d["norm_weight"])
    q, gate = (xn @ d["q_proj_weight"].t()).reshape(tokens, heads, 512).split(256, dim=-1)
    k, v = ((xn @ d[n].t()).reshape(tokens, kvh, 256) for n in ("k_proj_weight", "v_proj_weight"))
    pos = torch.arange(start, start + tokens, device=x.device)

    def rope(y):
        freq = theta ** (-torch.arange(0, rope_dim, 2, dtype=torch.float64, device=y.device) / rope_dim)
        cs, sn = ((pos.double()[:, None] * freq).cos()[:, None], (pos.double()[:, None] * freq).sin()[:, None])
        out, h = y.clone(), rope_dim // 2
        ia, ib = (slice(0, rope_dim, 2), slice(1, rope_dim, 2)) if interleaved else (slice(0, h), slice(h, rope_dim))
        out[..., ia], out[..., ib] = y[..., ia] * cs - y[..., ib] * sn, y[..., ia] * sn + y[..., ib] * cs
        return out

    q, k = rope(norm(q, d["q_norm_weight"])), rope(norm(k, d["k_norm_weight"]))
    keys, values = kc.double(), vc.double()
    keys[start:start + tokens], values[start:start + tokens] = k, v
    n = start + tokens
    dead = torch.arange(n, device=x.device)[None] > pos[:, None]
    o = torch.stack([torch.softmax((q[:, h] @ keys[:n, h * kvh // heads].t() / 16.0).masked_fill(dead, -torch.inf), -1)
                     @ values[:n, h * kvh // heads] for h in range(heads)], 1)
    return (o * torch.sigmoid(gate)).reshape(tokens, -1) @ d["out_proj_weight"].t(), k, v


# rows: a row block's edges (64 / G tokens), one call of a few rows (the
# decode entry), many; contexts: none, inside a tile, several chunks
@pytest.mark.parametrize("tokens,start,hidden,heads,kvh,x_dtype,cache_dtype,interleaved", [
    (5, 0, 2048, 16, 2, torch.float32, torch.float32, True),
    (8, 37, 512, 8, 1, torch.bfloat16, torch.float32, True),
    (32, 300, 2048, 16, 2, torch.float32, torch.bfloat16, True),
    (33, 0, 2048, 16, 2, torch.float32, torch.float32, False),
    (65, 15, 1024, 4, 4, torch.bfloat16, torch.bfloat16, True),
    (200, 1000, 2048, 16, 2, torch.float32, torch.float32, True),
    (131, 777, 512, 8, 4, torch.float32, torch.bfloat16, False),
    # either side of the decode entry's line for few heads
    (9, 40, 512, 8, 1, torch.float32, torch.float32, True),
    (10, 40, 512, 8, 1, torch.float32, torch.float32, True),
    (17, 200, 2048, 2, 1, torch.bfloat16, torch.float32, True),
    (18, 200, 2048, 2, 1, torch.bfloat16, torch.float32, True),
    (8, 21, 1536, 12, 3, torch.float32, torch.bfloat16, True),
])
def test_prompt_rows(tokens, start, hidden, heads, kvh, x_dtype, cache_dtype, interleaved):
    x, kc, vc, w = _inputs(tokens, tokens, hidden, heads, kvh, start + tokens + 3, x_dtype, cache_dtype)
    kw = dict(start_position=start, attention_heads=heads, kv_heads=kvh, rope_dim=64, rope_theta=1e4, rope_interleaved=interleaved)
    update, k2, v2 = hip.hip_qwen36_batched_attention_decode(x, kc, vc, *w.values(), **kw)
    ref, k, v = _reference(x, kc, vc, w, start, heads, kvh, 64, 1e4, interleaved)
    # 32-bit products and sums; the RoPE angles are 32-bit (2^-24 of the position)
    tol = 2e-6 + (start + tokens) * 2.0 ** -24 * 0.5
    assert float((update.double() - ref).norm() / ref.norm()) < tol
    rows = slice(start, start + tokens)
    rtol = (4e-3 if cache_dtype == torch.bfloat16 else 1e-6) + (start + tokens) * 2.0 ** -23
    for got, want, old in ((k2, k, kc), (v2, v, vc)):
        assert torch.allclose(got[rows].double(), want, rtol=rtol, atol=rtol)
        assert torch.equal(got[:start], old[:start]) and torch.equal(got[start + tokens:], old[start + tokens:])
    again = hip.hip_qwen36_batched_attention_decode(x, kc, vc, *w.values(), **kw)
    assert torch.equal(update, again[0])


def _error(seed, tokens, start, hidden, heads, kvh, cache_dtype, q_norm=1.0):
    """Relative error against float64 without rotation (whose 32-bit angles are
    the largest part of it otherwise) and with q norm weights near 1 + q_norm
    (scores of a few units, as a trained model's)."""

    x, kc, vc, w = _inputs(seed, tokens, hidden, heads, kvh, start + tokens, torch.float32, cache_dtype)
    w["q_norm_weight"] = (w["q_norm_weight"].float() + q_norm).bfloat16()
    got = hip.hip_qwen36_batched_attention_decode(
        x, kc, vc, *w.values(), start_position=start, attention_heads=heads, kv_heads=kvh, rope_dim=0)[0]
    ref, _, _ = _reference(x, kc, vc, w, start, heads, kvh, 0, 1e4, True)
    return float((got.double() - ref).norm() / ref.norm())


def test_long_prompt_in_calls_of_bounded_size():
    """2,100 rows: three calls on one workspace that no longer prompt grows, as
    one call of the C entry (a single chunk of positions per workgroup) gives."""

    tokens, start = 2100, 5
    x, kc, vc, w = _inputs(12, tokens, 512, 16, 2, start + tokens, torch.float32, torch.float32)
    hip._workspaces.clear()
    update, k, v = hip.hip_qwen36_batched_attention_decode(x, kc, vc, *w.values(), start_position=start)
    lib = _lib.load()
    kept = [t.numel() for (kind, _, _), t in hip._workspaces.items() if kind == "attention_prompt"]
    assert kept == [lib.fk_attention_prompt_workspace_bytes(1024, 512, 16, 2, 256, 1, 1)]
    ref, rk, _ = _reference(x, kc, vc, w, start, 16, 2, 64, 1e4, True)
    tol = 2e-6 + tokens * 2.0 ** -24 * 0.5  # (as test_prompt_rows)
    assert float((update.double() - ref).norm() / ref.norm()) < tol
    assert torch.allclose(k[start:].double(), rk, rtol=tokens * 2.0 ** -23, atol=tokens * 2.0 ** -23)

    one, k2, v2 = torch.empty_like(update), kc.clone(), vc.clone()
    n = lib.fk_attention_prompt_workspace_bytes(tokens, 512, 16, 2, 256, 1, 1)
    ws = torch.zeros(n, dtype=torch.uint8, device="cuda")
    p = {name: t.data_ptr() for name, t in w.items()}
    _lib.call("fk_attention_prompt", x.data_ptr(), 0, p["norm_weight"], 1, p["q_proj_weight"], p["k_proj_weight"],
              p["v_proj_weight"], p["out_proj_weight"], 1, p["q_norm_weight"], p["k_norm_weight"], 1, k2.data_ptr(),
              v2.data_ptr(), 0, start + tokens, start, tokens, 512, 16, 2, 256, 64, 1e4, 1, 1e-6, 1e-6, one.data_ptr(),
              None, ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream)
    assert float((one.double() - ref).norm() / ref.norm()) < tol
    # (sums over K in the same steps whatever the tile: the last bits of the larger tiles aside)
    assert torch.allclose(k2, k, rtol=1e-4, atol=1e-5) and torch.allclose(v2, v, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("tokens", [700, 1030])
def test_long_prompt_residual(tokens):
    """The layer's hidden states, written by the larger tiles of the output
    projection (700 rows: K unsplit; a second call of 6)."""

    x, kc, vc, w = _inputs(13, tokens, 2048, 16, 2, tokens, torch.bfloat16, torch.float32)
    gen = torch.Generator().manual_seed(14)
    moe = [_randn(gen, s, 0.02) for s in ((2048,), (16, 2048), (16, 128, 2048), (16, 2048, 64), (128, 2048), (2048, 64), (2048,))]
    _, hidden, update, *_ = hip.hip_qwen36_batched_attention_moe_layer_decode(x, kc, vc, *w.values(), *moe, top_k=2)
    ref, _, _ = _reference(x, kc, vc, w, 0, 16, 2, 64, 1e4, True)
    assert float((update.double() - ref).norm() / ref.norm()) < 2e-6 + tokens * 2.0 ** -24 * 0.5
    assert torch.equal(hidden, x.float() + update)


# A score is a sum of 256 products, whose roundings all reach the output.  In
# short chains added in pairs, as the dot products of few rows are (4 products
# and 6 levels), the variance is about 8 to 12 squared roundings of the score;
# in two chains of 128 products it is 64.  Measured: 3.1e-7 to 4.6e-7 and
# 6.1e-7 to 9.9e-7; the bound lies between them.
@pytest.mark.parametrize("tokens,start,hidden,heads,kvh,cache_dtype", [
    (8, 1000, 512, 8, 1, torch.float32),
    (32, 3000, 512, 16, 2, torch.bfloat16),
    (200, 1000, 2048, 16, 2, torch.float32),
])
def test_prompt_sums_are_as_exact_as_dot_products(tokens, start, hidden, heads, kvh, cache_dtype):
    errs = [_error(seed, tokens, start, hidden, heads, kvh, cache_dtype) for seed in range(3)]
    assert sum(errs) / 3 < 5.2e-7, errs


# step calls with long chunks of positions per workgroup (64, 32, 21 and 16
# chunks for 1 to 4 tokens): the last chunk length of the loop over tiles (48)
# and the first past it, tiles of 64 positions with every kind of remainder,
# a last chunk of own positions, of few positions and an empty one, groups of
# 2 and 4 query heads
@pytest.mark.parametrize("tokens,start,hidden,heads,kvh,cache_dtype", [
    (1, 3071, 2048, 16, 2, torch.float32),
    (1, 3072, 2048, 16, 2, torch.float32),
    (1, 3527, 2048, 16, 2, torch.bfloat16),
    (1, 4095, 2048, 16, 2, torch.bfloat16),
    (1, 4096, 2048, 16, 2, torch.float32),
    (2, 2100, 2048, 16, 2, torch.float32),
    (3, 1640, 2048, 16, 2, torch.bfloat16),
    (4, 1037, 2048, 16, 2, torch.float32),
    (4, 12000, 2048, 16, 2, torch.float32),
    (1, 12000, 2048, 16, 2, torch.bfloat16),
    (1, 9000, 2048, 16, 8, torch.float32),
])
def test_step_of_long_chunks(tokens, start, hidden, heads, kvh, cache_dtype):
    test_prompt_rows(tokens, start, hidden, heads, kvh, torch.float32, cache_dtype, True)


def test_long_chunk_sums_are_as_exact_as_the_loop_over_tiles():
    """Scores in chains of four products and values in sums of four positions,
    as the loop over tiles adds them (4.96e-7 here): 5.10e-7.  In chains of
    eight, with the values on the running sum: 5.50e-7."""

    errs = [_error(seed, 4, 12000, 512, 16, 2, torch.float32, 3.0) for seed in range(8)]
    assert sum(errs) / 8 < 5.3e-7, errs


def test_rows_see_no_later_row():
    """A later row that is not finite, or just other, changes no earlier row."""

    x, kc, vc, w = _inputs(3, 40, 512, 8, 1, 90, torch.float32, torch.float32)
    kw = dict(start_position=50, attention_heads=8, kv_heads=1, rope_dim=64)
    good = hip.hip_qwen36_batched_attention_decode(x, kc, vc, *w.values(), **kw)[0]
    bad = x.clone()
    bad[21], bad[30:] = float("nan"), 3.0
    got = hip.hip_qwen36_batched_attention_decode(bad, kc, vc, *w.values(), **kw)[0]
    assert torch.equal(got[:21], good[:21])
    assert bool(got[21:].isnan().all())


@pytest.mark.parametrize("tokens", [8, 17])
def test_decode_workspace_off_the_16_byte_boundary(tokens):
    """fk_attention_decode asks no alignment of its workspace beyond 8 bytes."""

    x, kc, vc, w = _inputs(9, tokens, 2048, 16, 2, 400, torch.float32, torch.float32)
    names = {"norm_weight": "input_norm_weight", "out_proj_weight": "o_proj_weight"}
    plan = AttentionStepPlan({names.get(k, k): v for k, v in w.items()}, tokens, max_positions=400, hidden=x)
    outs = []
    for offset in (0, 8):
        size = plan.workspace.numel()
        store = torch.zeros(size + 4096, dtype=torch.uint8, device="cuda")
        plan.workspace = store[offset:offset + size]
        plan.key_cache.copy_(kc)
        plan.value_cache.copy_(vc)
        plan.set_position(300)
        plan.run()
        outs.append(plan.update.clone())
        assert int(store[offset + size:].sum()) == 0
    assert bool(outs[0].isfinite().all()) and torch.equal(*outs)


# the single launch, the four launches and the matrix products
@pytest.mark.parametrize("tokens", [1, 4, 6, 8, 32])
@pytest.mark.parametrize("position", [-1, 61, 2**31 - 1])
def test_device_position_past_the_cache(tokens, position):
    """Also where position + tokens passes the range of an int: NaN, caches
    untouched, the position left where it is and flagged."""

    x, kc, _, w = _inputs(8, tokens, 2048, 16, 2, 61, torch.bfloat16, torch.float32)
    names = {"norm_weight": "input_norm_weight", "out_proj_weight": "o_proj_weight"}
    plan = AttentionStepPlan({names.get(k, k): v for k, v in w.items()}, tokens, max_positions=61, hidden=x)
    plan.key_cache.copy_(kc)
    plan.set_position(position)
    plan.run()
    torch.cuda.synchronize()
    assert bool(plan.update.isnan().all()) and int(plan.position) == position
    assert torch.equal(plan.key_cache, kc)
    with pytest.raises(_lib.FastKernelsError) as info:
        plan.check_device()
    assert info.value.status == _lib.FK_ERR_DEVICE


@pytest.mark.parametrize("tokens,start,row", [(8, 1000, 0), (8, 30, 7), (40, 100, 17), (70, 0, 69)])
def test_infinite_value_of_the_call_stays_infinite(tokens, start, row):
    """One value of one row overflows: the rows that see it get that infinity,
    in that dim alone, and the rows before it nothing."""

    x, kc, vc, w = _inputs(4, tokens, 512, 16, 2, start + tokens, torch.float32, torch.float32)
    x[:, 3], x[row, 3] = 0.0, 5.0
    w["norm_weight"][3] = 0.0
    w["v_proj_weight"][5], w["v_proj_weight"][5, 3] = 0.0, 3e38  # kv head 0, dim 5
    w["out_proj_weight"][:, 5:8 * 256:256] = 0.02               # of its eight query heads: the infinities add up
    kw = dict(start_position=start, attention_heads=16, kv_heads=2, rope_dim=64)
    got, _, v = hip.hip_qwen36_batched_attention_decode(x, kc, vc, *w.values(), **kw)
    assert bool(v[start + row, 0, 5].isposinf()) and int((~v.isfinite()).sum()) == 1
    assert bool(got[row:].isposinf().all())
    w["v_proj_weight"][5, 3] = 0.0
    assert torch.equal(got[:row], hip.hip_qwen36_batched_attention_decode(x, kc, vc, *w.values(), **kw)[0][:row])


# the last cached position before the step's own (one that loads past the
# chunk repeat), and an inner one, for calls of few and of many rows
@pytest.mark.parametrize("tokens,start,at", [(1, 4095, 4094), (1, 4095, 70), (3, 3071, 3070), (4, 12000, 11999), (8, 1000, 999), (33, 900, 31)])
def test_infinite_cached_value_stays_infinite(tokens, start, at):
    x, kc, vc, w = _inputs(5, tokens, 512, 16, 2, start + tokens, torch.float32, torch.float32)
    vc[at, 0, 5] = float("inf")
    w["out_proj_weight"][:, 5:8 * 256:256] = 0.02
    got = hip.hip_qwen36_batched_attention_decode(
        x, kc, vc, *w.values(), start_position=start, attention_heads=16, kv_heads=2, rope_dim=64)[0]
    assert bool(got.isposinf().all())


@pytest.mark.parametrize("tokens", [8, 32])
def test_device_position_advances_and_is_checked(tokens):
    x, kc, vc, w = _inputs(7, tokens, 2048, 16, 2, 4 * tokens, torch.bfloat16, torch.float32)
    names = {"norm_weight": "input_norm_weight", "out_proj_weight": "o_proj_weight"}
    plan = AttentionStepPlan({names.get(k, k): v for k, v in w.items()}, tokens, max_positions=4 * tokens - 1, hidden=x)
    plan.run()
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        plan.run(stream)
    graph.replay()
    graph.replay()
    assert int(plan.position) == 3 * tokens
    plan.check_device()
    spec = plan.spec
    k, v = torch.zeros_like(plan.key_cache), torch.zeros_like(plan.value_cache)
    for step in range(3):
        update, k, v = hip.hip_qwen36_batched_attention_decode(
            x, k, v, *w.values(), start_position=step * tokens, rope_theta=spec.rope_theta)
    assert torch.equal(plan.key_cache, k) and torch.allclose(plan.update, update, rtol=1e-4, atol=1e-5)
    graph.replay()  # past the cache: NaN, caches untouched, position left, flagged
    torch.cuda.synchronize()
    assert bool(plan.update.isnan().all()) and int(plan.position) == 3 * tokens and torch.equal(plan.key_cache, k)
    with pytest.raises(_lib.FastKernelsError) as info:
        plan.check_device()
    assert info.value.status == _lib.FK_ERR_DEVICE


def test_entry_refuses_what_it_does_not_take():
    lib = _lib.load()
    assert lib.fk_attention_prompt_workspace_bytes(40, 2048, 16, 2, 128, 1, 1) == 0
    assert lib.fk_attention_prompt_workspace_bytes(40, 2048, 16, 2, 256, 0, 1) == 0
    assert lib.fk_attention_prompt_workspace_bytes(0, 2048, 16, 2, 256, 1, 1) == 0
    assert lib.fk_attention_prompt_workspace_bytes(40, 2048, 16, 2, 256, 1, 1) > 0

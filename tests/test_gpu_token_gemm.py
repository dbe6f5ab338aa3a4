"""Projections of token batches on the matrix cores, against float64.

A value enters the products as three bf16 terms (24 bits), so the error is
that of fp32: each product is exact to 2^-24 of |w| |x|, and the sum over K
adds at most K / 64 + 6 roundings of 2^-24 of a partial sum of |w| |x|.  The
bound below, (K / 64 + 16) * 2^-24 * sum |w| |x (1 + n)| * rs, covers both, the
norm's scale and the weight product.
"""

from __future__ import annotations

import pytest
import torch

from fastkernels_amd.kernels import hip

pytestmark = pytest.mark.gpu


def _randn(gen, shape, scale=1.0, dtype=torch.bfloat16):
    return (torch.randn(shape, generator=gen) * scale).to(dtype).cuda()


def _check(outs, x, norm, weights, eps=1e-6):
    xd = x.double()
    xn = xd * torch.rsqrt((xd * xd).mean(-1, keepdim=True) + eps) * (1.0 + norm.double())
    k = x.shape[1]
    for out, w in zip(outs, weights):
        ref = xn @ w.double().t()
        bound = (k / 64 + 16) * 2.0 ** -24 * (xn.abs() @ w.double().abs().t())
        assert out.shape == ref.shape and out.dtype == torch.float32
        assert bool(((out.double() - ref).abs() <= bound).all()), float(((out.double() - ref).abs() / bound).max())


# every tile (32, 64, 128 tokens; 64, 128, 256 rows), its edges, and row
# counts that end inside a tile; K = 64 is a single step
@pytest.mark.parametrize("tokens,hidden,rows,x_dtype", [
    (4, 64, (16, 32, 16), torch.float32),
    (10, 192, (48, 80, 16), torch.bfloat16),
    (33, 512, (8192, 4096, 32), torch.float32),
    (65, 2048, (8192, 4096, 32), torch.bfloat16),
    (129, 2048, (8192, 4096, 32), torch.float32),
    (257, 1024, (8192, 4096, 32), torch.float32),
    (400, 4096, (8192, 4096, 32), torch.float32),
    # either side of the rule's lines for few rows
    (11, 2048, (512, 256, 16), torch.float32),
    (12, 2048, (512, 256, 16), torch.bfloat16),
    (8, 1024, (512, 256, 16), torch.float32),
    (9, 1024, (512, 256, 16), torch.float32),
])
def test_deltanet_projection_batches(tokens, hidden, rows, x_dtype):
    gen = torch.Generator().manual_seed(tokens)
    x = _randn(gen, (tokens, hidden), 1.0, x_dtype)
    norm = _randn(gen, (hidden,), 0.1)
    w = [_randn(gen, (n, hidden), 0.02) for n in (rows[0], rows[1], rows[2], rows[2])]
    outs = hip.hip_qwen36_batched_deltanet_project(x, norm, *w, block_hidden=4096)
    _check(outs, x, norm, w)
    again = hip.hip_qwen36_batched_deltanet_project(x, norm, *w, block_hidden=4096)
    assert all(torch.equal(a, b) for a, b in zip(outs, again))


@pytest.mark.parametrize("tokens", [10, 11, 12, 40, 200])
def test_attention_projection_batches(tokens):
    gen = torch.Generator().manual_seed(tokens)
    x, norm = _randn(gen, (tokens, 2048), 1.0, torch.float32), _randn(gen, (2048,), 0.1)
    w = [_randn(gen, (n, 2048), 0.02) for n in (1024, 512, 512)]
    _check(hip.hip_qwen36_batched_attention_project(x, norm, *w), x, norm, w)


def test_large_and_non_finite_tokens():
    """A token near the largest float, and one with an infinity or a NaN: the
    other tokens' rows are untouched, the non-finite ones are NaN (0 * inf of
    the norm), as with the per-row products of smaller batches."""

    gen = torch.Generator().manual_seed(3)
    x, norm = _randn(gen, (20, 512), 1.0, torch.float32), _randn(gen, (512,), 0.1)
    x[3, 7], x[5, 100], x[9] = float("inf"), float("nan"), x[9] * 1e15
    w = [_randn(gen, (n, 512), 0.02) for n in (64, 32, 16, 16)]
    outs = hip.hip_qwen36_batched_deltanet_project(x, norm, *w)
    few = hip.hip_qwen36_batched_deltanet_project(x[3:6], norm, *w)
    for o, f in zip(outs, few):
        assert bool(o[3].isnan().all()) and bool(o[5].isnan().all()) and bool(f[0].isnan().all()) and bool(f[2].isnan().all())
    keep = [t for t in range(20) if t not in (3, 5)]
    _check([o[keep] for o in outs], x[keep], norm, w)


@pytest.mark.parametrize("tokens", [4, 40, 200])
def test_values_past_the_bf16_range(tokens):
    """A finite value above the largest bf16 (3.39e38) is no infinity: its
    token's norm scale is 0 (the squares overflow), and so are its products."""

    gen = torch.Generator().manual_seed(5)
    x, norm = _randn(gen, (tokens, 512), 1.0, torch.float32), _randn(gen, (512,), 0.1)
    norm[7] = 0.0
    x[2, 7], x[3, 7] = 3.4e38, -3.4028234e38
    w = [_randn(gen, (n, 512), 0.02) for n in (64, 32, 16, 16)]
    for out in hip.hip_qwen36_batched_deltanet_project(x, norm, *w):
        assert bool((out[2:4] == 0).all()) and bool(out.isfinite().all())


@pytest.mark.parametrize("tokens", [13, 70, 300])
def test_outputs_off_the_16_byte_boundary(tokens):
    """The C entry's outputs need no alignment: the same values one float at a time."""

    from fastkernels_amd import _lib

    gen = torch.Generator().manual_seed(tokens)
    x, norm = _randn(gen, (tokens, 512), 1.0, torch.float32), _randn(gen, (512,), 0.1)
    w = [_randn(gen, (n, 512), 0.02) for n in (4096, 512, 512)]
    want = hip.hip_qwen36_batched_attention_project(x, norm, *w)
    stores = [torch.full((tokens * n.shape[0] + 2,), 7.0, device="cuda") for n in w]
    _lib.call("fk_attention_project", x.data_ptr(), 0, norm.data_ptr(), 1, *(t.data_ptr() for t in w), 1, tokens, 512, 4096,
              512, 1e-6, 1.0, *(t[1:].data_ptr() for t in stores), torch.cuda.current_stream().cuda_stream)
    for store, o in zip(stores, want):
        assert torch.equal(store[1:-1].view_as(o), o) and float(store[0]) == 7.0 and float(store[-1]) == 7.0

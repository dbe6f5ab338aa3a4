"""The DeltaNet operators at the edges of their token blocks: the conv's rows
of 8, the recurrence's chunks of 16, head_dim 128 (the scan kernel) and 64
(the general one)."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from fastkernels_amd.kernels import hip

pytestmark = pytest.mark.gpu


def _randn(gen, shape, scale=1.0, dtype=torch.float32):
    return (torch.randn(shape, generator=gen) * scale).to(dtype)


@pytest.mark.parametrize("kernel_size", [1, 4, 8])
@pytest.mark.parametrize("tokens", [1, 3, 8, 9, 24, 37])
def test_conv_blocks(tokens, kernel_size):
    gen = torch.Generator().manual_seed(tokens * 10 + kernel_size)
    channels = 300  # ends inside a workgroup
    mixed, state = _randn(gen, (tokens, channels)), _randn(gen, (channels, kernel_size))
    w = _randn(gen, (channels, 1, kernel_size))
    out, nxt = hip.hip_qwen36_batched_deltanet_conv(mixed.cuda(), state.cuda(), w.cuda())
    comb = torch.cat((state, mixed.t()), dim=1)
    ref = F.silu(F.conv1d(comb.double()[None, :, 1:], w.double(), groups=channels)[0]).t()
    # KS products and sums of values below ~5, and the exponential's last bits
    assert torch.allclose(out.cpu().double(), ref, rtol=1e-5, atol=kernel_size * 25 * 2.0 ** -23)
    assert torch.equal(nxt.cpu(), comb[:, -kernel_size:])


@pytest.mark.parametrize("tokens,qk_heads,value_heads,head_dim", [
    (1, 16, 32, 128), (15, 2, 4, 128), (16, 4, 4, 128), (17, 16, 32, 128), (32, 1, 2, 128), (51, 16, 32, 128),
    (19, 2, 4, 64),
])
def test_recurrence_chunks(tokens, qk_heads, value_heads, head_dim):
    gen = torch.Generator().manual_seed(tokens)
    hidden, vw = 256, value_heads * head_dim
    args = dict(
        mixed_qkv=_randn(gen, (tokens, 2 * qk_heads * head_dim + vw)), z=_randn(gen, (tokens, vw)),
        a_logits=_randn(gen, (tokens, value_heads)), b_logits=_randn(gen, (tokens, value_heads)),
        recurrent_state=_randn(gen, (value_heads, head_dim, head_dim), 0.1),
        out_proj_weight=_randn(gen, (hidden, vw), 0.02, torch.bfloat16), linear_norm_weight=_randn(gen, (head_dim,)),
        a_log=_randn(gen, (value_heads,), 0.5), dt_bias=_randn(gen, (value_heads,), 0.5),
    )
    dev = {k: v.cuda() for k, v in args.items()}
    update, state = hip.hip_qwen36_batched_deltanet_recurrent_output(
        *dev.values(), qk_heads=qk_heads, value_heads=value_heads, head_dim=head_dim)

    d = {k: v.double() for k, v in args.items()}
    q, k, v = d["mixed_qkv"].split((qk_heads * head_dim, qk_heads * head_dim, vw), dim=-1)
    rep = value_heads // qk_heads
    unit = lambda x: x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q = unit(q.reshape(tokens, qk_heads, head_dim)).repeat_interleave(rep, 1) * head_dim ** -0.5
    k = unit(k.reshape(tokens, qk_heads, head_dim)).repeat_interleave(rep, 1)
    v = v.reshape(tokens, value_heads, head_dim)
    decay = torch.exp(-d["a_log"].exp() * F.softplus(d["a_logits"] + d["dt_bias"]))
    beta = torch.sigmoid(d["b_logits"])
    s, core = d["recurrent_state"], []
    for t in range(tokens):
        s = s * decay[t][:, None, None]
        s = s + k[t][:, :, None] * ((v[t] - (s * k[t][:, :, None]).sum(1)) * beta[t][:, None])[:, None, :]
        core.append((s * q[t][:, :, None]).sum(1))
    o = torch.stack(core)
    o = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + 1e-6) * d["linear_norm_weight"] * F.silu(
        d["z"].reshape(tokens, value_heads, head_dim))
    ref = o.reshape(tokens, vw) @ d["out_proj_weight"].t()
    # 32-bit states: every token adds a few 2^-24 of the state's size, which
    # its decay and delta forget again
    assert float((state.cpu().double() - s).norm() / s.norm()) < 2e-6
    assert float((update.cpu().double() - ref).norm() / ref.norm()) < 4e-6

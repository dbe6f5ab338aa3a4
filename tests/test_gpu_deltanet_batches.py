"""The DeltaNet operators at the edges of their token blocks: the conv's rows
of 8, the recurrence's chunks of 16, head_dim 128 (the scan kernel) and 64
(the general one), and the step call at the sizes between its launches."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from fastkernels_amd.kernels import hip

pytestmark = pytest.mark.gpu


def _randn(gen, shape, scale=1.0, dtype=torch.float32):
    return (torch.randn(shape, generator=gen) * scale).to(dtype)


def test_conv_in_place():
    """The C entry with its outputs over its inputs gives what separate ones give."""

    from fastkernels_amd import _lib

    gen = torch.Generator().manual_seed(5)
    mixed, state, w = (_randn(gen, s).cuda() for s in ((37, 300), (300, 4), (300, 1, 4)))
    out, nxt = hip.hip_qwen36_batched_deltanet_conv(mixed, state, w)
    _lib.call("fk_deltanet_conv", mixed.data_ptr(), 0, state.data_ptr(), 0, w.data_ptr(), 0, 37, 300, 4,
              mixed.data_ptr(), state.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert torch.equal(mixed, out) and torch.equal(state, nxt)


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


def test_conv_of_more_blocks_than_a_grid_dimension_holds():
    """524,281 rows and more are over 65,535 blocks of 8: the blocks grow."""

    gen = torch.Generator().manual_seed(6)
    mixed, state, w = _randn(gen, (524_300, 3)), _randn(gen, (3, 4)), _randn(gen, (3, 1, 4))
    out, nxt = hip.hip_qwen36_batched_deltanet_conv(mixed.cuda(), state.cuda(), w.cuda())
    comb = torch.cat((state, mixed.t()), dim=1)
    ref = F.silu(F.conv1d(comb.double()[None, :, 1:], w.double(), groups=3)[0]).t()
    assert torch.allclose(out.cpu().double(), ref, rtol=1e-5, atol=4 * 25 * 2.0 ** -23)
    assert torch.equal(nxt.cpu(), comb[:, -4:])


@pytest.mark.parametrize("state_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens", [3, 20, 97, 128])
def test_recurrence_in_place_and_bf16_states(tokens, state_dtype):
    """The C entry with the next state over the state, of either type (the scan
    and the chunks), and with outputs off the 16-byte boundary, gives what
    separate ones give; a bf16 state is read exactly and rounds once."""

    from fastkernels_amd import _lib

    gen = torch.Generator().manual_seed(tokens)
    mixed, z = _randn(gen, (tokens, 2 * 2 * 128 + 512)).cuda(), _randn(gen, (tokens, 512)).cuda()
    a, b = _randn(gen, (tokens, 4)).cuda(), _randn(gen, (tokens, 4)).cuda()
    state = _randn(gen, (4, 128, 128), 0.1).to(state_dtype).cuda()
    rest = [_randn(gen, (256, 512), 0.02, torch.bfloat16).cuda(), *(_randn(gen, s).cuda() for s in ((128,), (4,), (4,)))]
    run = lambda s: hip.hip_qwen36_batched_deltanet_recurrent_output(  # noqa: E731
        mixed, z, a, b, s, *rest, qk_heads=2, value_heads=4, head_dim=128)
    update, after = run(state)
    update32, after32 = run(state.float())
    assert after.dtype == state_dtype and torch.equal(update, update32) and torch.equal(after, after32.to(state_dtype))
    import ctypes
    codes = (ctypes.c_int32 * 10)(0, 0, 0, 0, 0 if state_dtype == torch.float32 else 1, 1, 0, 0, 0, 0)
    n = _lib.load().fk_deltanet_workspace_bytes(tokens, 4, 128)
    ws = torch.zeros(n, dtype=torch.uint8, device="cuda")
    store = torch.zeros(2 * tokens * 256 + 8, device="cuda")
    residual = _randn(gen, (tokens, 256)).cuda()
    got, out = store[1:1 + tokens * 256], store[3 + tokens * 256:3 + 2 * tokens * 256]  # 4 and 12 bytes past a boundary
    _lib.call("fk_deltanet_recurrent_output", *(t.data_ptr() for t in (mixed, z, a, b, state, *rest, residual)),
              ctypes.cast(codes, ctypes.c_void_p), tokens, 2, 4, 128, 256, 1e-6, got.data_ptr(), state.data_ptr(),
              out.data_ptr(), ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream)
    assert torch.equal(got.view(tokens, 256), update) and torch.equal(state, after)
    assert torch.equal(out.view(tokens, 256), residual + update)


@pytest.mark.parametrize("tokens,qk_heads,value_heads,head_dim", [
    (2, 16, 32, 128), (3, 16, 32, 128), (15, 2, 4, 128), (16, 4, 4, 128), (17, 16, 32, 128), (32, 1, 2, 128), (51, 16, 32, 128),
    (19, 2, 4, 64), (95, 2, 4, 128), (96, 1, 5, 128), (97, 2, 4, 128), (112, 16, 32, 128), (127, 1, 2, 128), (100, 4, 4, 128),
    (250, 2, 4, 128),
])
@pytest.mark.parametrize("hidden", [256, 250])  # 250: the general output projection
def test_recurrence_chunks(tokens, qk_heads, value_heads, head_dim, hidden):
    gen = torch.Generator().manual_seed(tokens)
    vw = value_heads * head_dim
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


@pytest.mark.parametrize("what", ["value", "key", "beta"])
def test_recurrence_keeps_a_non_finite_token_from_earlier_ones(what):
    """Rows before a non-finite token (inside a chunk of 16) are what they are without it, other heads' states too."""

    tokens, bad, gen = 120, 101, torch.Generator().manual_seed(1)
    mixed, z = _randn(gen, (tokens, 2 * 2 * 128 + 512)).cuda(), _randn(gen, (tokens, 512)).cuda()
    a, b, state = _randn(gen, (tokens, 4)).cuda(), _randn(gen, (tokens, 4)).cuda(), _randn(gen, (4, 128, 128), 0.1).cuda()
    rest = (_randn(gen, (256, 512), 0.02, torch.bfloat16).cuda(), _randn(gen, (128,)).cuda(), _randn(gen, (4,), 0.5).cuda(),
            _randn(gen, (4,), 0.5).cuda())
    run = lambda: hip.hip_qwen36_batched_deltanet_recurrent_output(  # noqa: E731
        mixed, z, a, b, state, *rest, qk_heads=2, value_heads=4, head_dim=128)
    update, after = run()
    if what == "value":
        mixed[bad, 512 + 3] = float("inf")  # head 0, column 3
    elif what == "key":
        mixed[bad, 256 + 5] = float("nan")  # qk head 0: value heads 0 and 1
    else:
        b[bad, 0] = float("nan")
    update2, after2 = run()
    # (that chunk goes token by token: a delta may round once more or less, 2^-24 of values below 4)
    near = lambda x, y: torch.allclose(x, y, rtol=1e-6, atol=4e-6)  # noqa: E731
    assert near(update2[:bad], update[:bad])
    assert not torch.isfinite(update2[bad]).any() and not torch.isfinite(after2[0]).all()
    assert torch.equal(after2[2:], after[2:])
    if what == "value":  # the state's other columns too
        keep = [c for c in range(128) if c != 3]
        assert near(after2[0][:, keep], after[0][:, keep]) and torch.equal(after2[1], after[1])


@pytest.mark.parametrize("tokens", [20, 97, 100, 112])
def test_recurrence_infinite_last_value(tokens):
    """An infinite value of the last token leaves its column of the state
    infinite (k times it), also where the last chunk of 16 is not full."""

    gen = torch.Generator().manual_seed(2)
    mixed, z = _randn(gen, (tokens, 2 * 2 * 128 + 512)), _randn(gen, (tokens, 512))
    mixed[-1, 512 + 3] = float("inf")  # head 0, column 3
    a, b, state = _randn(gen, (tokens, 4)), _randn(gen, (tokens, 4)), _randn(gen, (4, 128, 128), 0.1)
    rest = (_randn(gen, (256, 512), 0.02, torch.bfloat16), _randn(gen, (128,)), _randn(gen, (4,), 0.5), _randn(gen, (4,), 0.5))
    _, after = hip.hip_qwen36_batched_deltanet_recurrent_output(
        *(t.cuda() for t in (mixed, z, a, b, state, *rest)), qk_heads=2, value_heads=4, head_dim=128)
    column = after[0, :, 3].cpu()
    assert bool(column.isinf().all()) and torch.equal(column > 0, mixed[-1, 256:384] > 0)
    assert int((~after.isfinite()).sum()) == 128


@pytest.mark.parametrize("tokens,conv_dtype", [(9, torch.bfloat16), (16, torch.bfloat16), (33, torch.float32),
                                               (64, torch.bfloat16), (4, torch.float32)])
def test_step_equals_staged_operators(tokens, conv_dtype):
    """fk_deltanet_step past its single launch runs the staged kernels: the
    same values as the operators one by one, and the same on a second call."""

    from fastkernels_amd.plan import DeltaNetStepPlan
    from fastkernels_amd.workloads import make_deltanet_weights

    w = make_deltanet_weights(seed=tokens, device="cuda")
    w["conv_state"] = w["conv_state"].to(conv_dtype)
    x = _randn(torch.Generator().manual_seed(1), (tokens, 2048)).cuda()
    plan = DeltaNetStepPlan(w, tokens, hidden=x)
    for _ in range(2):
        plan.run()
    plan.check_device()
    mixed, z, a, b = hip.hip_qwen36_batched_deltanet_project(
        x, w["input_norm_weight"], w["in_proj_qkv_weight"], w["in_proj_z_weight"], w["in_proj_a_weight"], w["in_proj_b_weight"])
    mixed, conv = hip.hip_qwen36_batched_deltanet_conv(mixed, w["conv_state"], w["conv1d_weight"])
    update, rec = hip.hip_qwen36_batched_deltanet_recurrent_output(
        mixed, z, a, b, w["recurrent_state"], w["out_proj_weight"], w["linear_norm_weight"], w["a_log"], w["dt_bias"])
    assert torch.equal(plan.next_conv_state, conv) and torch.equal(plan.next_recurrent_state, rec)
    assert torch.equal(plan.update, update) and torch.equal(plan.hidden_out, x + update)

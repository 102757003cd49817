"""GPU parity of the causal depthwise convolution kernels (C ABI: rglru_hip_conv_fwd / _bwd) against the
oracle's restatement of griffin/griffin.py:474-487 and autograd through it."""

import pytest
import torch

from oracle import rglru_oracle as orc
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu

FP32_TOL = 1e-5     # norm-wise relative, fp32 storage
BF16_TOL = 2e-2     # bf16 storage, fp32 arithmetic, against the fp32 oracle on the bf16-rounded inputs


def _say(*args):
    print(*args, flush=True)


def _positions(B, T, kind, seed):
    """Token positions: one document continued from earlier calls, fresh documents, or several
    documents packed into each row."""
    if kind == "continued":
        return torch.arange(5, 5 + T).repeat(B, 1)
    if kind == "fresh":
        return torch.arange(T).repeat(B, 1)
    g = torch.Generator().manual_seed(seed)
    pos = torch.empty(B, T, dtype=torch.long)
    for b in range(B):
        p = int(torch.randint(0, 4, (1,), generator=g))
        for t in range(T):
            if t > 0 and float(torch.rand(1, generator=g)) < 0.15:
                p = 0
            pos[b, t] = p
            p += 1
    return pos


def _case(B, T, W, K, seed, with_state, with_bias):
    g = torch.Generator().manual_seed(seed)
    u = torch.randn(B, T, W, generator=g)
    w = torch.randn(W, K, generator=g) * (1.0 / K) ** 0.5
    b = torch.randn(W, generator=g) * 0.1 if with_bias else None
    state = torch.randn(B, K - 1, W, generator=g) if with_state else None
    dout = torch.randn(B, T, W, generator=g)
    return u, w, b, state, dout


def _oracle(u, w, b, state, dout, pos, dtype):
    def prep(t):
        return None if t is None else t.to(dtype).to(torch.float32).requires_grad_(True)
    u_, w_, b_, s_ = prep(u), prep(w), prep(b), prep(state)
    B, T, W = u.shape
    K = w.shape[1]
    out, new_state = orc.causal_conv(u_, w_, torch.zeros(W) if b_ is None else b_,
                                     torch.zeros(B, K - 1, W) if s_ is None else s_, pos)
    leaves = [t for t in (u_, w_, b_, s_) if t is not None]
    grads = torch.autograd.grad(out, leaves, dout.to(dtype).to(torch.float32))
    names = [n for n, t in zip(("u", "w", "b", "state"), (u_, w_, b_, s_)) if t is not None]
    return out.detach(), new_state.detach(), dict(zip(names, grads))


def _hip(u, w, b, state, dout, pos, dtype):
    from griffin_amd.hip_block_ops import hip_causal_conv

    def prep(t):
        return None if t is None else t.to(dtype).cuda().requires_grad_(True)
    u_, b_, s_ = prep(u), prep(b), prep(state)
    w_ = w.to(dtype)[:, None, :].contiguous().cuda().requires_grad_(True)
    out, new_state = hip_causal_conv(u_, s_, w_, b_, pos.cuda())
    leaves = [t for t in (u_, w_, b_, s_) if t is not None]
    grads = list(torch.autograd.grad(out, leaves, dout.to(dtype).cuda()))
    torch.cuda.synchronize()
    names = [n for n, t in zip(("u", "w", "b", "state"), (u_, w_, b_, s_)) if t is not None]
    grads[1] = grads[1][:, 0, :]
    return out.detach(), new_state.detach(), dict(zip(names, grads))


CASES = [
    # B, T, W, K, positions, carried state, bias
    (2, 50, 64, 4, "packed", True, True),      # vector path, several documents per row
    (2, 37, 24, 4, "packed", True, True),      # fp32 rows of 96 bytes (vector path), bf16 rows of 48 (vector path)
    (3, 33, 13, 4, "packed", True, True),      # odd width: one element per thread
    (1, 2, 64, 4, "continued", True, True),    # shorter than the kernel: the new state mixes old state and input
    (2, 100, 128, 3, "fresh", False, True),    # three taps, no carried state
    (2, 40, 32, 2, "continued", True, False),  # two taps, no bias
    (2, 19, 16, 1, "packed", False, True),     # a single tap: a per-channel scale and shift
    (4, 300, 256, 4, "packed", True, True),    # several runs per sequence, halo across run boundaries
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("cfg", CASES)
def test_conv_matches_oracle(cfg, dtype):
    B, T, W, K, kind, with_state, with_bias = cfg
    _say("conv case", cfg, dtype)
    u, w, b, state, dout = _case(B, T, W, K, seed=3, with_state=with_state, with_bias=with_bias)
    pos = _positions(B, T, kind, seed=4)
    want_out, want_state, want_g = _oracle(u, w, b, state, dout, pos, dtype)
    got_out, got_state, got_g = _hip(u, w, b, state, dout, pos, dtype)
    tol = FP32_TOL if dtype == torch.float32 else BF16_TOL
    errs = {"out": rel_err(got_out.float(), want_out)}
    for name in want_g:
        errs["d" + name] = rel_err(got_g[name].float(), want_g[name])
    _say("  rel errors:", {k: "%.2e" % v for k, v in errs.items()})
    for name, err in errs.items():
        assert err < tol, (name, err)
    # the carried state is a copy of input rows: exact in the storage type
    assert torch.equal(got_state.float().cpu(), want_state.to(dtype).float())


def test_conv_split_equals_one_pass_at_training_shape():
    """B8 T2048 W1024 bf16: the sequence convolved in three pieces with the carried state equals one
    pass bit for bit (each output depends on the same K rows either way), and the input gradient is
    linear in the upstream gradient."""
    from griffin_amd.hip_block_ops import hip_causal_conv

    g = torch.Generator().manual_seed(9)
    B, T, W, K = 8, 2048, 1024, 4
    u = torch.randn(B, T, W, generator=g).bfloat16().cuda()
    w = (torch.randn(W, 1, K, generator=g) * 0.5).bfloat16().cuda()
    b = (torch.randn(W, generator=g) * 0.1).bfloat16().cuda()
    pos = torch.arange(T).repeat(B, 1).cuda()
    pos[3, 700:] -= 700
    whole, last = hip_causal_conv(u, None, w, b, pos)
    pieces, state, start = [], None, 0
    for stop in (5, 1031, T):
        piece, state = hip_causal_conv(u[:, start:stop].contiguous(), state, w, b, pos[:, start:stop].contiguous())
        pieces.append(piece)
        start = stop
    assert torch.equal(torch.cat(pieces, dim=1), whole)
    assert torch.equal(state, last)
    uu = u.clone().requires_grad_(True)
    out, _ = hip_causal_conv(uu, None, w, b, pos)
    d1 = torch.randn(B, T, W, generator=g).bfloat16().cuda()
    g1, = torch.autograd.grad(out, uu, d1, retain_graph=True)
    g2, = torch.autograd.grad(out, uu, 2 * d1)
    torch.cuda.synchronize()
    assert rel_err(g2.float(), 2 * g1.float()) < 1e-2


def test_conv_argument_errors():
    from griffin_amd.hip_block_ops import hip_causal_conv

    u = torch.randn(2, 8, 16, device="cuda")
    w = torch.randn(16, 1, 4, device="cuda")
    pos = torch.arange(8, device="cuda").repeat(2, 1)
    with pytest.raises(RuntimeError):
        hip_causal_conv(u.cpu(), None, w.cpu(), None, pos.cpu())
    with pytest.raises(ValueError):
        hip_causal_conv(u, None, torch.randn(16, 1, 9, device="cuda"), None, pos)      # kernel size beyond the maximum
    with pytest.raises(ValueError):
        hip_causal_conv(u, torch.zeros(2, 2, 16, device="cuda"), w, None, pos)         # state of the wrong length
    with pytest.raises(ValueError):
        hip_causal_conv(u, None, w, None, pos[:, :4])
    with pytest.raises(TypeError):
        hip_causal_conv(u.double(), None, w.double(), None, pos)


# ----------------------------------------------------------------------------------------------
# output gate h * gelu_tanh(v) (C ABI: rglru_hip_gelu_gate_fwd / _bwd)
# ----------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(2, 50, 64), (3, 7, 13), (1, 1, 1), (4, 300, 256), (5, 1023)])
def test_gelu_gate_matches_oracle(shape, dtype):
    from griffin_amd.hip_block_ops import hip_gelu_gate

    _say("gelu gate case", shape, dtype)
    g = torch.Generator().manual_seed(11)
    h = torch.randn(*shape, generator=g) * 1.5
    v = torch.randn(*shape, generator=g) * 3.0          # covers the saturated tails of tanh
    dout = torch.randn(*shape, generator=g)
    hr = h.to(dtype).float().requires_grad_(True)
    vr = v.to(dtype).float().requires_grad_(True)
    want = orc.gelu_gate(hr, vr)
    want_dh, want_dv = torch.autograd.grad(want, (hr, vr), dout.to(dtype).float())
    hh = h.to(dtype).cuda().requires_grad_(True)
    vh = v.to(dtype).cuda().requires_grad_(True)
    got = hip_gelu_gate(hh, vh)
    got_dh, got_dv = torch.autograd.grad(got, (hh, vh), dout.to(dtype).cuda())
    torch.cuda.synchronize()
    tol = FP32_TOL if dtype == torch.float32 else BF16_TOL
    errs = {"out": rel_err(got.float(), want), "dh": rel_err(got_dh.float(), want_dh), "dv": rel_err(got_dv.float(), want_dv)}
    _say("  rel errors:", {k: "%.2e" % e for k, e in errs.items()})
    for name, err in errs.items():
        assert err < tol, (name, err)


def test_gelu_gate_special_values_at_training_shape():
    """B8 T2048 W1024 bf16: exact zeros where either factor is zero, the identity far in the positive
    tail, zero far in the negative tail, and linearity in h."""
    from griffin_amd.hip_block_ops import hip_gelu_gate

    g = torch.Generator().manual_seed(12)
    shape = (8, 2048, 1024)
    h = torch.randn(*shape, generator=g).bfloat16().cuda()
    v = (torch.randn(*shape, generator=g) * 2).bfloat16().cuda()
    assert torch.count_nonzero(hip_gelu_gate(h, torch.zeros_like(v))) == 0
    assert torch.count_nonzero(hip_gelu_gate(torch.zeros_like(h), v)) == 0
    big = torch.full_like(v, 40.0)
    assert torch.equal(hip_gelu_gate(h, big), (h.float() * 40.0).bfloat16())
    assert torch.count_nonzero(hip_gelu_gate(h, -big)) == 0
    out1 = hip_gelu_gate(h, v).float()
    out2 = hip_gelu_gate(2 * h, v).float()
    assert rel_err(out2, 2 * out1) < 1e-2


def test_gelu_gate_argument_errors():
    from griffin_amd.hip_block_ops import hip_gelu_gate

    a = torch.randn(4, 8, device="cuda")
    with pytest.raises(RuntimeError):
        hip_gelu_gate(a.cpu(), a.cpu())
    with pytest.raises(ValueError):
        hip_gelu_gate(a, a[:, :4])
    with pytest.raises(TypeError):
        hip_gelu_gate(a, a.bfloat16())
    with pytest.raises(TypeError):
        hip_gelu_gate(a.double(), a.double())


# ----------------------------------------------------------------------------------------------
# convolution over right-padded batches (C ABI: rglru_hip_conv_padded_fwd)
# ----------------------------------------------------------------------------------------------
def _padded_inputs(B, T, W, K, seed, pattern):
    g = torch.Generator().manual_seed(seed)
    u = torch.randn(B, T, W, generator=g)
    w = torch.randn(W, K, generator=g) * (1.0 / K) ** 0.5
    b = torch.randn(W, generator=g) * 0.1
    state = torch.randn(B, K - 1, W, generator=g)
    if pattern == "right":                                   # rows of different lengths, padded on the right
        lengths = torch.randint(0, T + 1, (B,), generator=g)
        lengths[0] = T
        if B > 1:
            lengths[1] = 0                                   # an empty row: state must pass through
        active = torch.arange(T)[None, :] < lengths[:, None]
    elif pattern == "mixed":                                 # right-padded rows and rows with holes side by side:
        lengths = torch.randint(0, T + 1, (B,), generator=g)  # the two kinds go to different kernels of one call
        active = torch.arange(T)[None, :] < lengths[:, None]
        active[::2] = torch.rand((B + 1) // 2, T, generator=g) > 0.3
    else:                                                    # holes anywhere
        active = torch.rand(B, T, generator=g) > 0.3
    pos = _positions(B, T, "packed", seed + 1)
    return u, w, b, state, pos, active


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("cfg", [(3, 50, 64, 4, "right"), (4, 200, 24, 4, "holes"), (2, 130, 13, 3, "holes"),
                                 (3, 65, 128, 2, "right"), (2, 7, 16, 1, "holes"), (5, 300, 64, 4, "mixed"),
                                 (4, 2100, 256, 4, "right")])
def test_padded_conv_matches_oracle(cfg, dtype):
    from griffin_amd.hip_block_ops import hip_causal_conv_padded

    B, T, W, K, pattern = cfg
    _say("padded conv case", cfg, dtype)
    u, w, b, state, pos, active = _padded_inputs(B, T, W, K, seed=13, pattern=pattern)
    up = lambda t: t.to(dtype).float()
    want, want_state = orc.causal_conv_padded(up(u), up(w), up(b), up(state), pos, active)
    got, got_state = hip_causal_conv_padded(u.to(dtype).cuda(), state.to(dtype).cuda(),
                                            w.to(dtype)[:, None, :].contiguous().cuda(), b.to(dtype).cuda(),
                                            pos.cuda(), active.cuda())
    torch.cuda.synchronize()
    tol = FP32_TOL if dtype == torch.float32 else BF16_TOL
    err = rel_err(got.float(), want)
    _say("  rel error:", "%.2e" % err)
    assert err < tol
    assert torch.count_nonzero(got[~active.cuda()]) == 0
    # the carried window is made of copies of input or state rows (or zeros): exact in the storage type
    assert torch.equal(got_state.float().cpu(), want_state.to(dtype).float())


def test_padded_conv_all_active_equals_dense_kernel_at_training_shape():
    """B8 T2048 W1024 bf16, every token active, documents starting at position 0: the padded kernel
    and the dense kernel walk the same K rows per output and agree bit for bit."""
    from griffin_amd.hip_block_ops import hip_causal_conv, hip_causal_conv_padded

    g = torch.Generator().manual_seed(17)
    B, T, W, K = 8, 2048, 1024, 4
    u = torch.randn(B, T, W, generator=g).bfloat16().cuda()
    w = (torch.randn(W, 1, K, generator=g) * 0.5).bfloat16().cuda()
    b = (torch.randn(W, generator=g) * 0.1).bfloat16().cuda()
    pos = torch.arange(T).repeat(B, 1).cuda()
    pos[5, 1000:] -= 1000
    active = torch.ones(B, T, dtype=torch.bool, device="cuda")
    dense, _ = hip_causal_conv(u, None, w, b, pos)
    padded, _ = hip_causal_conv_padded(u, None, w, b, pos, active)
    assert torch.equal(dense, padded)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("cfg", [(3, 50, 64, 4, "right"), (4, 200, 24, 4, "holes"), (2, 130, 13, 3, "holes"),
                                 (3, 65, 128, 2, "right"), (2, 7, 16, 1, "holes"), (2, 300, 1024, 4, "holes"),
                                 (5, 300, 64, 4, "mixed"), (4, 700, 256, 3, "right")])
def test_padded_conv_gradients_match_oracle_autograd(cfg, dtype):
    """Reverse mode of the padded convolution (C ABI: rglru_hip_conv_padded_bwd) against autograd through
    the oracle's token-by-token loop: gradients at the input, the carried state, the taps and the bias."""
    from griffin_amd.hip_block_ops import hip_causal_conv_padded

    B, T, W, K, pattern = cfg
    _say("padded conv gradient case", cfg, dtype)
    u, w, b, state, pos, active = _padded_inputs(B, T, W, K, seed=29, pattern=pattern)
    dout = torch.randn(B, T, W, generator=torch.Generator().manual_seed(31))
    up = lambda t: t.to(dtype).float()
    ref = [up(t).clone().requires_grad_(True) for t in (u, w, b, state)]
    want, _ = orc.causal_conv_padded(ref[0], ref[1], ref[2], ref[3], pos, active)
    want.backward(up(dout))
    dev = [u.to(dtype).cuda().requires_grad_(True), w.to(dtype)[:, None, :].contiguous().cuda().requires_grad_(True),
           b.to(dtype).cuda().requires_grad_(True), state.to(dtype).cuda().requires_grad_(True)]
    got, _ = hip_causal_conv_padded(dev[0], dev[3], dev[1], dev[2], pos.cuda(), active.cuda())
    got.backward(dout.to(dtype).cuda())
    torch.cuda.synchronize()
    tol = FP32_TOL if dtype == torch.float32 else BF16_TOL
    names = ("input", "taps", "bias", "state")
    for name, r, d in zip(names, ref, dev):
        if K == 1 and name == "state":
            continue
        grad = d.grad.float().cpu().reshape(r.grad.shape)
        err = rel_err(grad, r.grad)
        _say("  d%s rel error: %.2e" % (name, err))
        assert err < tol, name
    # padding receives no gradient at all
    assert torch.count_nonzero(dev[0].grad[~active.cuda()]) == 0


# ----------------------------------------------------------------------------------------------
# RMSNorm in front of the block (C ABI: rglru_hip_rmsnorm_fwd / _bwd)
# ----------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(2, 50, 64), (3, 7, 13), (1, 1, 768), (4, 33, 1024), (2, 5, 2560), (300, 24),
                                   (70, 4096), (9, 5000), (33, 8192)])
def test_rmsnorm_matches_oracle(shape, dtype):
    from griffin_amd.hip_block_ops import hip_rmsnorm

    from griffin_amd.hip_block_ops import rmsnorm_max_width

    _say("rmsnorm case", shape, dtype)
    if shape[-1] > rmsnorm_max_width(dtype):
        pytest.skip("wider than one wave holds in this storage type: the module uses the portable operators there")
    gen = torch.Generator().manual_seed(21)
    x = torch.randn(*shape, generator=gen) * 1.7 + 0.3
    scale = torch.randn(shape[-1], generator=gen) * 0.2
    dy = torch.randn(*shape, generator=gen)
    xr = x.to(dtype).float().requires_grad_(True)
    sr = scale.to(dtype).float().requires_grad_(True)
    want = orc.rmsnorm(xr, sr)
    want_dx, want_dg = torch.autograd.grad(want, (xr, sr), dy.to(dtype).float())
    xh = x.to(dtype).cuda().requires_grad_(True)
    sh = scale.to(dtype).cuda().requires_grad_(True)
    got = hip_rmsnorm(xh, sh)
    got_dx, got_dg = torch.autograd.grad(got, (xh, sh), dy.to(dtype).cuda())
    torch.cuda.synchronize()
    tol = FP32_TOL if dtype == torch.float32 else BF16_TOL
    errs = {"y": rel_err(got.float(), want), "dx": rel_err(got_dx.float(), want_dx), "dg": rel_err(got_dg.float(), want_dg)}
    _say("  rel errors:", {k: "%.2e" % e for k, e in errs.items()})
    for name, err in errs.items():
        assert err < tol, (name, err)


def test_rmsnorm_module_and_properties_at_training_shape():
    """B8 T2048 D768 bf16 through the module: rows leave with mean square (1 + g)^2-weighted ~ 1 for a
    zero scale, a positive rescaling of the input changes nothing (eps aside), and the module's state
    dict keeps the reference's single parameter name."""
    from griffin_amd import RMSNorm

    norm = RMSNorm(768).cuda().bfloat16()
    assert list(norm.state_dict()) == ["g"]
    gen = torch.Generator().manual_seed(22)
    x = (torch.randn(8, 2048, 768, generator=gen) * 3).bfloat16().cuda()
    y = norm(x)
    ms = y.float().pow(2).mean(-1)
    assert (ms - 1.0).abs().max().item() < 2e-2
    y4 = norm(4 * x)                                          # a power of two: exact in bf16
    assert rel_err(y4.float(), y.float()) < 1e-2
    with pytest.raises(ValueError):
        from griffin_amd.hip_block_ops import hip_rmsnorm
        hip_rmsnorm(x, torch.zeros(5, device="cuda", dtype=torch.bfloat16))


# ----------------------------------------------------------------------------------------------
# sum of the partial weight gradients of a split contraction (C ABI: rglru_hip_sum_sets)
# ----------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(8, 2048, 768), (16, 768, 1024), (3, 7, 13), (1, 64, 64), (9, 1, 5), (2, 1000001)])
def test_sum_sets_matches_a_float64_sum(shape, dtype):
    from griffin_amd.hip_block_ops import _sum_sets

    _say("sum of sets", shape, dtype)
    x = torch.randn(*shape, generator=torch.Generator().manual_seed(41)).to(dtype)
    want = x.double().sum(0)
    got = _sum_sets(x.cuda())
    torch.cuda.synchronize()
    assert got.dtype == dtype and got.shape == want.shape
    # fp32 accumulation, one rounding to the storage type
    tol = 1e-6 if dtype == torch.float32 else 4e-3
    assert rel_err(got.double(), want) < tol
    # a view that is not contiguous takes the generic reduction and still agrees
    strided = x.cuda().transpose(0, 1) if x.dim() == 3 else None
    if strided is not None:
        assert rel_err(_sum_sets(strided).double(), x.double().transpose(0, 1).sum(0)) < tol


def test_sum_sets_rejects_bad_arguments():
    from griffin_amd import _lib

    lib = _lib.load()
    buf = torch.zeros(64, device="cuda")
    assert lib.rglru_hip_sum_sets(buf.data_ptr(), buf.data_ptr(), 0, 8, 0, None) != 0
    assert lib.rglru_hip_sum_sets(None, buf.data_ptr(), 2, 8, 0, None) != 0
    assert lib.rglru_hip_sum_sets(buf.data_ptr(), buf.data_ptr(), 2, 8, 7, None) != 0


# ----------------------------------------------------------------------------------------------
# bias gradient of the block's Linear layers (C ABI: rglru_hip_colsum)
# ----------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(2, 50, 64, 96), (3, 7, 13, 5), (1, 1, 768, 1024), (8, 2048, 768, 1024), (2, 129, 24, 1030)])
def test_hip_linear_matches_torch_linear(shape, dtype):
    """Output and all three gradients of hip_linear against torch.nn.functional.linear in fp64 on the same
    (rounded) operands; the bias gradient is the column sum the library computes."""
    from griffin_amd.hip_block_ops import hip_linear

    B, T, D, W = shape
    _say("linear case", shape, dtype)
    gen = torch.Generator().manual_seed(33)
    x = torch.randn(B, T, D, generator=gen).to(dtype)
    w = (torch.randn(W, D, generator=gen) / D ** 0.5).to(dtype)
    b = (torch.randn(W, generator=gen) * 0.1).to(dtype)
    dy = torch.randn(B, T, W, generator=gen).to(dtype)
    ref = [t.double().requires_grad_(True) for t in (x, w, b)]
    torch.nn.functional.linear(*ref).backward(dy.double())
    dev = [t.cuda().requires_grad_(True) for t in (x, w, b)]
    out = hip_linear(*dev)
    out.backward(dy.cuda())
    torch.cuda.synchronize()
    tol = 2e-5 if dtype == torch.float32 else BF16_TOL
    want = torch.nn.functional.linear(x.double(), w.double(), b.double())
    assert rel_err(out.double().cpu(), want) < tol
    for name, r, d in zip(("x", "weight", "bias"), ref, dev):
        err = rel_err(d.grad.double().cpu(), r.grad)
        _say("  d%s rel error: %.2e" % (name, err))
        assert err < tol, name


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(2, 50, 64, 96), (3, 7, 13, 5), (8, 2048, 768, 1024)])
@pytest.mark.parametrize("used", ["both", "first", "second"])
def test_hip_linear_pair_matches_two_linear_layers(shape, dtype, used):
    """The block's two input projections as one autograd node (griffin/griffin.py:462-464): outputs and all
    five gradients against two torch.nn.functional.linear calls in fp64, also when only one of the two
    outputs takes part in the loss."""
    from griffin_amd.hip_block_ops import hip_linear_pair

    B, T, D, W = shape
    _say("linear pair case", shape, dtype, used)
    gen = torch.Generator().manual_seed(34)
    x = torch.randn(B, T, D, generator=gen).to(dtype)
    ws = [(torch.randn(W, D, generator=gen) / D ** 0.5).to(dtype) for _ in range(2)]
    bs = [(torch.randn(W, generator=gen) * 0.1).to(dtype) for _ in range(2)]
    dys = [torch.randn(B, T, W, generator=gen).to(dtype) for _ in range(2)]
    take = [used in ("both", "first"), used in ("both", "second")]
    ref = [t.double().requires_grad_(True) for t in (x, ws[0], bs[0], ws[1], bs[1])]
    outs = (torch.nn.functional.linear(ref[0], ref[1], ref[2]), torch.nn.functional.linear(ref[0], ref[3], ref[4]))
    sum((o * d.double()).sum() for o, d, t in zip(outs, dys, take) if t).backward()
    dev = [t.cuda().requires_grad_(True) for t in (x, ws[0], bs[0], ws[1], bs[1])]
    got = hip_linear_pair(*dev)
    sum((o.float() * d.cuda().float()).sum() for o, d, t in zip(got, dys, take) if t).backward()
    torch.cuda.synchronize()
    tol = 2e-5 if dtype == torch.float32 else BF16_TOL
    for o, w in zip(got, outs):
        assert rel_err(o.double().cpu(), w.detach()) < tol
    for name, r, d in zip(("x", "w1", "b1", "w2", "b2"), ref, dev):
        if r.grad is None:
            assert d.grad is None, name
            continue
        err = rel_err(d.grad.double().cpu(), r.grad)
        _say("  d%s rel error: %.2e" % (name, err))
        assert err < tol, name


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(2, 50, 64, 3), (3, 37, 13, 4), (1, 1, 8, 2), (8, 2048, 1024, 4)])
def test_strided_gradient_outputs_equal_the_contiguous_ones(shape, dtype):
    """rglru_hip_conv_bwd with du_stride and rglru_hip_gelu_gate_bwd with dv_stride (C ABI): du and dv written as the
    column halves of one [B, T, 2 W + pad] matrix are bit for bit what the contiguous calls write, nothing else of
    that matrix is touched, and the other outputs do not change."""
    from griffin_amd import _lib
    from griffin_amd.hip_block_ops import _DTYPE_CODES, _dtype_code, _ptr, _stream_ptr

    B, T, W, K = shape
    _say("strided gradient outputs case", shape, dtype)
    lib = _lib.load()
    g = torch.Generator().manual_seed(35)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).cuda()
    u, dout, h, v, dgate = rnd(B, T, W), rnd(B, T, W), rnd(B, T, W), rnd(B, T, W) * 2, rnd(B, T, W)
    taps = (torch.randn(W, K, generator=g) * 0.4).to(dtype).cuda()
    pos = torch.arange(T).repeat(B, 1).cuda()
    pos[:, T // 2:] -= T // 2                                 # a document start in the middle of every row
    code, stream = _dtype_code(dtype), _stream_ptr(u.device)
    pad = 8 if W % 8 == 0 else 3                              # rows of whole 16-byte vectors where W allows the vector kernels
    ld = 2 * W + pad

    def conv_bwd(du):
        scratch = torch.empty(lib.rglru_hip_conv_scratch_bytes(B, T, W, K), dtype=torch.uint8, device="cuda")
        dtaps = torch.empty(W, K, dtype=dtype, device="cuda")
        dbias = torch.empty(W, dtype=dtype, device="cuda")
        _lib.check(lib.rglru_hip_conv_bwd(_ptr(u), None, _ptr(taps), _ptr(pos), _ptr(dout), _ptr(scratch), _ptr(du), du.stride(1),
                                          None, _ptr(dtaps), _ptr(dbias), B, T, W, K, code, _DTYPE_CODES[dtype], _DTYPE_CODES[dtype],
                                          stream), "rglru_hip_conv_bwd")
        return dtaps, dbias

    def gate_bwd(dv):
        dh = torch.empty_like(h)
        _lib.check(lib.rglru_hip_gelu_gate_bwd(_ptr(dgate), _ptr(h), _ptr(v), _ptr(dh), _ptr(dv), h.numel(), W, dv.stride(1),
                                               code, stream), "rglru_hip_gelu_gate_bwd")
        return dh

    du_c, dv_c = torch.empty_like(u), torch.empty_like(v)
    want_conv, want_dh = conv_bwd(du_c), gate_bwd(dv_c)
    both = torch.full((B, T, ld), 7.0, dtype=dtype, device="cuda")
    got_conv, got_dh = conv_bwd(both[..., :W]), gate_bwd(both[..., W:2 * W])
    torch.cuda.synchronize()
    assert torch.equal(both[..., :W], du_c)
    assert torch.equal(both[..., W:2 * W], dv_c)
    assert torch.all(both[..., 2 * W:] == 7.0)
    assert torch.equal(got_dh, want_dh)
    for a, b in zip(got_conv, want_conv):
        assert torch.equal(a, b)
    # a stride below the width is an error, not a memory fault
    with pytest.raises(ValueError):
        _lib.check(lib.rglru_hip_gelu_gate_bwd(_ptr(dgate), _ptr(h), _ptr(v), _ptr(torch.empty_like(h)), _ptr(dv_c), h.numel(), W, W - 1,
                                               code, stream), "rglru_hip_gelu_gate_bwd")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(2, 50, 64, 96), (3, 7, 13, 5), (8, 2048, 768, 1024)])
def test_hip_linear_pair_with_stacked_gradients(shape, dtype):
    """The pair's backward when its two incoming gradients are the column halves of one matrix (what the
    one-launch block forward's backward hands it): one GEMM for dx, one for both weight gradients, one column
    sum -- against two torch.nn.functional.linear calls in fp64."""
    from griffin_amd.hip_block_ops import _stacked_halves, hip_linear_pair

    B, T, D, W = shape
    _say("linear pair, stacked gradients, case", shape, dtype)
    gen = torch.Generator().manual_seed(36)
    x = torch.randn(B, T, D, generator=gen).to(dtype)
    ws = [(torch.randn(W, D, generator=gen) / D ** 0.5).to(dtype) for _ in range(2)]
    bs = [(torch.randn(W, generator=gen) * 0.1).to(dtype) for _ in range(2)]
    both = torch.randn(B, T, 2 * W, generator=gen).to(dtype)
    ref = [t.double().requires_grad_(True) for t in (x, ws[0], bs[0], ws[1], bs[1])]
    outs = (torch.nn.functional.linear(ref[0], ref[1], ref[2]), torch.nn.functional.linear(ref[0], ref[3], ref[4]))
    torch.autograd.backward(outs, [both[..., :W].double(), both[..., W:].double()])
    dev = [t.cuda().requires_grad_(True) for t in (x, ws[0], bs[0], ws[1], bs[1])]
    got = hip_linear_pair(*dev)
    both_d = both.cuda()
    halves = [both_d[..., :W], both_d[..., W:]]
    assert _stacked_halves(*halves) is not None
    torch.autograd.backward(got, halves)
    torch.cuda.synchronize()
    tol = 2e-5 if dtype == torch.float32 else BF16_TOL
    for name, r, d in zip(("x", "w1", "b1", "w2", "b2"), ref, dev):
        err = rel_err(d.grad.double().cpu(), r.grad)
        _say("  d%s rel error: %.2e" % (name, err))
        assert err < tol, name


# ----------------------------------------------------------------------------------------------
# convolution + RG-LRU + output gate in one forward launch (rglru_hip_block_fwd), griffin/griffin.py:464-520
# ----------------------------------------------------------------------------------------------
def _block_case(B, T, W, nb, K, kind, carried, strided, seed):
    """Operands of the block between its projections, bf16 on the GPU."""
    torch.manual_seed(seed)
    bw = W // nb
    bf = torch.bfloat16

    def rnd(*shape, scale=1.0):
        return (scale * torch.randn(*shape)).to(bf).cuda()

    p = {"w_a": rnd(nb, bw, bw, scale=bw ** -0.5), "b_a": rnd(nb, bw), "w_x": rnd(nb, bw, bw, scale=bw ** -0.5),
         "b_x": rnd(nb, bw), "weight": rnd(W, 1, K, scale=0.4), "bias": rnd(W, scale=0.1)}
    # decays of 0.9 .. 0.999 per token at an open gate, as the reference initialises them: the state then
    # carries across many tiles, so a wrong carry between tiles shows
    p["lam"] = torch.logit(torch.empty(W).uniform_(0.9, 0.999).pow(1.0 / 8.0)).to(bf).cuda()
    if strided:                                       # the two projections as halves of one wider buffer
        both = rnd(B, T, 2 * W + 16)
        p["u"], p["v"] = both[..., :W], both[..., W + 16:]
    else:
        p["u"], p["v"] = rnd(B, T, W), rnd(B, T, W)
    p["conv_state"] = rnd(B, K - 1, W) if (carried and K > 1) else None
    p["h0"] = torch.randn(B, W).cuda() if carried else None
    p["pos"] = _positions(B, T, kind, seed).cuda()
    return p


def _three_kernels(p):
    """The same computation as three launches through the autograd wrappers of the separate kernels."""
    from griffin_amd.hip_block_ops import hip_causal_conv, hip_gelu_gate
    from griffin_amd.hip_scan import hip_rglru

    x, new_conv = hip_causal_conv(p["u"], p["conv_state"], p["weight"], p["bias"], p["pos"])
    y, h_last = hip_rglru(x, p["w_a"], p["b_a"], p["w_x"], p["b_x"], p["lam"], 8.0, p["h0"], p["pos"] == 0, None)
    return hip_gelu_gate(y, p["v"].contiguous()), h_last, new_conv


BLOCK_FWD_CASES = [
    # B, T, W, nb, K, positions, carried state, strided rows
    (2, 128, 256, 2, 4, "fresh", False, False),
    (3, 200, 256, 2, 4, "packed", True, False),
    (3, 67, 128, 2, 4, "continued", True, True),
    (2, 1, 128, 4, 4, "continued", True, False),
    (2, 2, 128, 4, 3, "packed", True, False),
    (5, 130, 192, 3, 2, "packed", True, True),
    (2, 64, 96, 3, 4, "packed", False, False),
    (4, 333, 64, 1, 1, "packed", True, False),
    (8, 2048, 1024, 8, 4, "fresh", False, False),
    (8, 2048, 1024, 16, 4, "packed", True, True),
]


@pytest.mark.parametrize("case", BLOCK_FWD_CASES)
def test_block_forward_matches_the_three_kernels(case):
    """One launch against conv_fwd + fwd + gelu_gate (each checked against the oracle above and in
    test_hip_gpu.py): the convolved rows and the carried rows are bit-identical, y and the gated output
    agree to the rounding of a carry composed in another order (see test_hip_gpu.py on reproducibility)."""
    from griffin_amd.hip_block_ops import hip_block_forward

    B, T, W, nb, K, kind, carried, strided = case
    p = _block_case(B, T, W, nb, K, kind, carried, strided, seed=B + T)
    _say("block forward", case)
    from griffin_amd.hip_scan import FIRST_TOKEN_RESET

    with torch.no_grad():
        want_gated, want_h, want_conv = _three_kernels(p)
        got_gated, got_h, got_conv = hip_block_forward(
            p["u"], p["v"], p["conv_state"], p["weight"], p["bias"], p["pos"],
            FIRST_TOKEN_RESET if (kind == "fresh" and not carried) else None,   # positions 0 .. T-1: no flag tensor
            p["w_a"], p["b_a"], p["w_x"], p["b_x"], p["lam"], p["h0"], 8.0)
    torch.cuda.synchronize()
    if K > 1:
        assert torch.equal(got_conv, want_conv)
    # one bf16 rounding step at the largest value is 2^-8 of it
    assert rel_err(got_gated.float().cpu(), want_gated.float().cpu()) < 5e-3
    assert rel_err(got_h.cpu(), want_h.cpu()) < 1e-5
    # a changed bit here and there, not a systematic difference
    differing = (got_gated != want_gated).float().mean().item()
    assert differing < 1e-3, differing


@pytest.mark.parametrize("case", BLOCK_FWD_CASES)
def test_block_forward_gradients_match_the_three_kernels(case):
    """Autograd through the one-launch forward (its backward runs gate, scan and convolution reverse kernels
    on the x and y the forward kept) against autograd through the three separate operators."""
    from griffin_amd.hip_block_ops import hip_block_flags, hip_block_forward
    from griffin_amd.hip_scan import FIRST_TOKEN_RESET

    B, T, W, nb, K, kind, carried, strided = case
    p = _block_case(B, T, W, nb, K, kind, carried, strided, seed=B + T)
    names = [n for n in ("u", "v", "conv_state", "weight", "bias", "w_a", "b_a", "w_x", "b_x", "lam", "h0") if p[n] is not None]
    dg = torch.randn(B, T, W).to(torch.bfloat16).cuda()
    dh = torch.randn(B, W).cuda()
    dc = torch.randn(B, K - 1, W).to(torch.bfloat16).cuda()   # a later call's gradient at the carried rows
    _say("block forward gradients", case)

    def grads(fused):
        q = dict(p)
        for n in names:
            q[n] = p[n].detach().clone().requires_grad_(True)
        if fused:
            gated, h_last, carried_rows = hip_block_forward(
                q["u"], q["v"], q["conv_state"], q["weight"], q["bias"], q["pos"],
                FIRST_TOKEN_RESET if (kind == "fresh" and not carried) else hip_block_flags(q["pos"]) if B % 2 else None,
                q["w_a"], q["b_a"], q["w_x"], q["b_x"], q["lam"], q["h0"], 8.0)
        else:
            gated, h_last, carried_rows = _three_kernels(q)
        outs, ups = [gated, h_last], [dg, dh]
        if K > 1:
            outs.append(carried_rows)
            ups.append(dc)
        return torch.autograd.grad(outs, [q[n] for n in names], ups)

    want, got = grads(False), grads(True)
    torch.cuda.synchronize()
    for n, a, b in zip(names, got, want):
        assert a.shape == b.shape and a.dtype == b.dtype, n
        assert rel_err(a.float().cpu(), b.float().cpu()) < 5e-3, n


def test_block_forward_random_shapes():
    """Forty seeded draws of batch, length, width, gate blocks, taps, position pattern, carried state and row
    strides: outputs and, for every second draw, gradients against the three separate operators."""
    import random

    from griffin_amd.hip_block_ops import hip_block_forward
    from griffin_amd.hip_scan import FIRST_TOKEN_RESET

    rng = random.Random(20)
    for trial in range(40):
        bw, nb = rng.choice([32, 64, 128]), rng.choice([1, 2, 3, 5, 8])
        B, T = rng.choice([1, 2, 3, 7]), rng.choice([1, 2, 3, 5, 31, 64, 65, 127, 128, 200, 257, 500])
        K, kind = rng.choice([1, 2, 3, 4]), rng.choice(["fresh", "continued", "packed"])
        carried, strided, with_grads = rng.random() < 0.5, rng.random() < 0.4, trial % 2 == 1
        _say("block forward draw", trial, (B, T, bw * nb, nb, K, kind, carried, strided, with_grads))
        p = _block_case(B, T, bw * nb, nb, K, kind, carried, strided, seed=trial)
        names = [n for n in ("u", "v", "weight", "bias", "w_a", "b_a", "w_x", "b_x", "lam") if p[n] is not None]
        marker = FIRST_TOKEN_RESET if (kind == "fresh" and not carried) else None

        def run(fused):
            q = dict(p)
            for n in names:
                q[n] = p[n].detach().clone().requires_grad_(with_grads)
            if fused:
                outs = hip_block_forward(q["u"], q["v"], q["conv_state"], q["weight"], q["bias"], q["pos"], marker,
                                         q["w_a"], q["b_a"], q["w_x"], q["b_x"], q["lam"], q["h0"], 8.0)
            else:
                outs = _three_kernels(q)
            got = [o.detach() for o in outs]
            if with_grads:
                ups = [torch.full_like(outs[0], 0.5), torch.ones_like(outs[1])]
                got += list(torch.autograd.grad(list(outs[:2]), [q[n] for n in names], ups))
            return got

        with torch.set_grad_enabled(with_grads):
            want, got = run(False), run(True)
        torch.cuda.synchronize()
        if K > 1:
            assert torch.equal(got[2], want[2]), trial
        for i, (a, b) in enumerate(zip(got, want)):
            assert a.shape == b.shape, (trial, i)
            if a.numel():                                    # one tap carries no rows
                assert rel_err(a.float().cpu(), b.float().cpu()) < 1e-2, (trial, i)


def test_block_forward_argument_errors():
    from griffin_amd import _lib
    from griffin_amd.hip_block_ops import hip_block_forward_covers

    assert hip_block_forward_covers(1024, 8, 4, torch.bfloat16)
    assert not hip_block_forward_covers(1024, 8, 4, torch.float32)      # 16-bit storage only
    assert not hip_block_forward_covers(2560, 8, 4, torch.bfloat16)     # blocks of 320 channels: three launches
    assert not hip_block_forward_covers(1024, 8, 5, torch.bfloat16)
    lib = _lib.load()
    buf = torch.zeros(1 << 16, device="cuda", dtype=torch.bfloat16)
    p = buf.data_ptr()
    args = [p, 0, p, 0, None, p, None, 4, 1, p, None, None, None, None, p, None, None, p, 2, 16, 128, 2, 1, None]
    bad_stride = list(args); bad_stride[1] = 64
    assert lib.rglru_hip_block_fwd(*bad_stride) != 0 and b"stride" in lib.rglru_hip_last_error()
    unaligned = list(args); unaligned[0] = p + 2
    assert lib.rglru_hip_block_fwd(*unaligned) != 0 and b"aligned" in lib.rglru_hip_last_error()
    wide = list(args); wide[20] = 640
    assert lib.rglru_hip_block_fwd(*wide) != 0


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.bfloat16, 1e-2)])
@pytest.mark.parametrize("rows,features,outputs", [(1, 8, 1), (16, 40, 17), (17, 104, 33), (33, 64, 16), (70, 1000, 2064), (129, 72, 4100)])
def test_decode_linear_matches_fp64(rows, features, outputs, dtype, tol):
    """The projections of a decode step at the edges of their tiles: row tiles of 16 to 64, column tiles of 16 and 32, a
    contraction that ends inside a step, rows of a wider buffer, rows that do not take part."""
    from griffin_amd import _lib
    from griffin_amd.hip_block_ops import _dtype_code, _ptr, _stream_ptr

    print("decode linear", rows, features, outputs, dtype, flush=True)
    torch.manual_seed(rows)
    wide = torch.randn(rows, features + 8, device="cuda", dtype=dtype)
    x = wide[:, :features]
    w = torch.randn(outputs, features, device="cuda", dtype=dtype) / features ** 0.5
    bias = torch.randn(outputs, device="cuda", dtype=dtype)
    active = (torch.arange(rows, device="cuda") % 3 != 1).to(torch.uint8)
    y = torch.empty(rows, outputs, device="cuda", dtype=dtype)
    _lib.check(_lib.load().rglru_hip_decode_linear(_ptr(x), x.stride(0), _ptr(w), _ptr(bias), _ptr(active), _ptr(y), rows,
                                                   outputs, features, _dtype_code(dtype), _stream_ptr(x.device)), "decode_linear")
    want = (x.double() @ w.double().t() + bias.double()) * active.double()[:, None]
    assert ((y.double() - want).norm() / want.norm()).item() < tol
    assert torch.count_nonzero(y[active == 0]).item() == 0


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.bfloat16, 1e-2)])
@pytest.mark.parametrize("features", [8, 16, 24, 32, 40])
def test_decode_linear_of_short_contractions(features, dtype, tol):
    """Contractions shorter than a step of the products (32 elements in bf16) and just beyond.  Values only: that the lanes past a row's
    end read inside the row is checked for every lane on the host (tests/test_cabi.py)."""
    from griffin_amd import _lib
    from griffin_amd.hip_block_ops import _dtype_code, _ptr, _stream_ptr

    print("decode linear, short", features, dtype, flush=True)
    gen = torch.Generator().manual_seed(features)
    x = torch.randn(3, features, generator=gen).to(dtype).cuda()
    w = torch.randn(64, features, generator=gen).to(dtype).cuda()
    y = torch.empty(3, 64, device="cuda", dtype=dtype)
    _lib.check(_lib.load().rglru_hip_decode_linear(_ptr(x), x.stride(0), _ptr(w), None, None, _ptr(y), 3, 64, features, _dtype_code(dtype),
                                                   _stream_ptr(x.device)), "decode_linear")
    want = x.double() @ w.double().t()
    assert ((y.double() - want).norm() / want.norm()).item() < tol


@pytest.mark.parametrize("blocks", [1, 3])
def test_decode_steps_of_blocks_of_16_channels(blocks):
    """Gate blocks of 16 channels fill half of a product's contraction.  Against the oracle, one step at a time and all of them in one
    launch; where the other half's lanes read is checked on the host (tests/test_cabi.py)."""
    from griffin_amd import PreparedParams, hip_rglru_step, hip_rglru_steps
    from oracle import rglru_oracle as orc
    from tests.helpers import PARAMS, oracle_run, rel_err

    print("decode steps of 16-wide blocks", blocks, flush=True)
    B, steps, W = 5, 3, 16 * blocks
    case = orc.make_case(B, steps, W, blocks, seed=blocks, h0_std=0.5, bias_std=0.5)
    want, last, _ = oracle_run(case, torch.bfloat16)
    prep = PreparedParams(*[case[k].bfloat16().cuda() for k in PARAMS[1:]], 8.0, torch.bfloat16)
    x = case["x"].bfloat16()
    state, state_at_once = case["h0"].cuda().contiguous(), case["h0"].cuda().contiguous()
    rows = [hip_rglru_step(x[:, t].contiguous().cuda(), prep, state) for t in range(steps)]
    at_once = hip_rglru_steps(x.transpose(0, 1).contiguous().cuda(), prep, state_at_once)
    for got, h in ((torch.stack(rows, 1), state), (at_once.transpose(0, 1), state_at_once)):
        assert rel_err(got.float(), want) < 2e-2 and rel_err(h, last) < 2e-2


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.bfloat16, 2e-2)])
@pytest.mark.parametrize("batch,dim,width,blocks,taps", [(1, 64, 128, 2, 4), (16, 40, 96, 3, 3), (17, 96, 160, 1, 2), (70, 72, 136, 2, 4), (130, 64, 64, 2, 1)])
def test_block_step_matches_the_library_route(batch, dim, width, blocks, taps, dtype, tol):
    """One token per row through the three launches of ``hip_block_step`` against the same block with the projections of
    the BLAS library and ``hip_block_decode_step`` (itself checked against the oracle), with inactive rows, document
    starts and a cache, and without any of them."""
    from griffin_amd import RecurrentBlock, RecurrentBlockCache, hip_block_ops

    print("block step", batch, dim, width, blocks, taps, dtype, flush=True)
    torch.manual_seed(batch)
    block = RecurrentBlock(dim, width, conv_kernel_size=taps, gate_blocks=blocks, scan_mode="hip").cuda().to(dtype).eval()
    with torch.no_grad():
        for name, p in block.named_parameters():
            if name.endswith("bias"):
                p.normal_(std=0.3)
        block.temporal_conv.weight.normal_(std=0.5)
        x = torch.randn(batch, 1, dim, device="cuda", dtype=dtype)
        cache = RecurrentBlockCache(torch.randn(batch, width, device="cuda"),
                                    torch.randn(batch, taps - 1, width, device="cuda", dtype=dtype),
                                    torch.arange(batch, device="cuda") % 5 - 1)
        active = (torch.arange(batch, device="cuda") % 4 != 2)[:, None]
        positions = (torch.arange(batch, device="cuda") % 3)[:, None]
        calls = [dict(), dict(cache=cache), dict(cache=cache, segment_pos=positions)]
        if batch > 2:
            calls += [dict(cache=cache, active_mask=active), dict(cache=cache, segment_pos=positions, active_mask=active)]
        real = hip_block_ops.hip_block_step
        for call in calls:
            got, got_cache = block(x, return_cache=True, **call)
            hip_block_ops.hip_block_step = lambda *args: None
            try:
                want, want_cache = block(x, return_cache=True, **call)
            finally:
                hip_block_ops.hip_block_step = real
            assert rel_err(got.float(), want.float()) < tol
            assert rel_err(got_cache.rnn_state, want_cache.rnn_state) < tol
            assert torch.equal(got_cache.segment_position, want_cache.segment_position)
            if taps > 1:
                assert rel_err(got_cache.conv_state.float(), want_cache.conv_state.float()) < tol


@pytest.mark.parametrize("B,T", [(1, 1), (3, 7), (2, 64), (4, 2047), (2, 2048), (3, 4100)])
@pytest.mark.parametrize("given,carried", [(False, False), (False, True), (True, True)])
def test_token_facts_match_the_elementwise_formulas(B, T, given, carried):
    """Positions, flag bytes, convolution positions, row words and last positions of one launch against the running counts
    they stand for, on rows that are whole, right-padded, empty and full of holes, over more than one pass of the kernel."""
    from griffin_amd.hip_block_ops import token_facts

    g = torch.Generator().manual_seed(B * 10000 + T)
    active = torch.rand(B, T, generator=g) < 0.7
    for b in range(B):
        if b % 4 == 1:
            active[b] = torch.arange(T) < max(T // 3, 1)
        elif b % 4 == 2:
            active[b] = False
        elif b % 4 == 3:
            active[b] = True
    prev = torch.randint(-1, 5, (B,), generator=g) if carried else None
    pos = torch.randint(0, 4, (B, T), generator=g) if given else None
    facts = token_facts(active.cuda(), None if pos is None else pos.cuda(), None if prev is None else prev.cuda())
    everything, prefix = facts.resolve()
    start = torch.full((B,), -1) if prev is None else prev
    want_pos = pos if given else start[:, None] + active.long().cumsum(1)
    assert torch.equal(facts.positions.cpu(), want_pos)
    want_last, rows = [], facts.rows.cpu()
    flags, conv = facts.flags.cpu(), facts.conv_positions.cpu()
    prefixes = []
    for b in range(B):
        order, doc, last = 0, -1, int(start[b])
        for t in range(T):
            a, p = bool(active[b, t]), int(want_pos[b, t])
            if a and p == 0:
                doc = order
            f = int(flags[b, t])
            assert (f & 1) == (p == 0) and ((f >> 1) & 1) == (not a)
            if a:
                hidden = 0 if doc < 0 else 3 - min(order - doc, 3)
                assert (f >> 2) == hidden, (b, t)
                assert int(conv[b, t]) == (1 << 30 if doc < 0 else order - doc)
                last = p
                order += 1
        want_last.append(last)
        prefixes.append(bool(active[b, :order].all()))
        assert rows[:, b].tolist() == [order, doc, int(prefixes[-1])]
    assert facts.last_position.tolist() == want_last
    assert everything == bool(active.all()) and prefix == all(prefixes)


@pytest.mark.parametrize("cfg", [(3, 70, 64, 128, 2, 4), (2, 129, 96, 256, 8, 3), (4, 64, 64, 192, 3, 2), (5, 33, 64, 64, 2, 1)])
@pytest.mark.parametrize("packed,carried", [(False, False), (True, False), (False, True), (True, True)])
def test_right_padded_block_in_one_launch_matches_the_separate_kernels(cfg, packed, carried):
    """A right-padded bf16 batch through the one-launch forward (flags with padding, row table in the backward convolution)
    against convolution, RG-LRU and gate as kernels of their own: output, cache and every gradient."""
    from griffin_amd import RecurrentBlock, RecurrentBlockCache

    B, T, D, W, blocks, taps = cfg
    print("padded block", cfg, packed, carried, flush=True)
    torch.manual_seed(T)
    block = RecurrentBlock(D, W, conv_kernel_size=taps, gate_blocks=blocks, scan_mode="hip").cuda().bfloat16()
    with torch.no_grad():
        for name, p in block.named_parameters():
            if name.endswith("bias"):
                p.normal_(std=0.2)
        block.temporal_conv.weight.normal_(std=0.5)
    x = torch.randn(B, T, D, device="cuda").bfloat16().requires_grad_(True)
    dy = torch.randn(B, T, D, device="cuda").bfloat16()
    lengths = torch.tensor([T, 1, T // 2, 0, T - 1][:B], device="cuda")
    token = torch.arange(T, device="cuda")
    active = token[None] < lengths[:, None]
    positions = (token[None] + 3 * torch.arange(B, device="cuda")[:, None]) % 19 if packed else None
    cache = None
    leaves = [x, *block.parameters()]
    if carried:
        cache = RecurrentBlockCache(torch.randn(B, W, device="cuda").requires_grad_(True),
                                    torch.randn(B, taps - 1, W, device="cuda").bfloat16().requires_grad_(True),
                                    torch.arange(B, device="cuda") + 1)
        leaves += [cache.rnn_state] + ([cache.conv_state] if taps > 1 else [])
    results = []
    for covers in (True, False):
        real = block._hip_block_forward_covers
        if not covers:
            block._hip_block_forward_covers = lambda *args: False
        try:
            out, new = block(x, cache, positions, active_mask=active, return_cache=True)
        finally:
            block._hip_block_forward_covers = real
        results.append((out, new, torch.autograd.grad(out, leaves, dy)))
    (a, na, ga), (b, nb, gb) = results
    assert torch.count_nonzero(a[~active]).item() == 0
    assert rel_err(a.float(), b.float()) < 1e-2
    assert rel_err(na.rnn_state, nb.rnn_state) < 1e-2 and torch.equal(na.segment_position, nb.segment_position)
    if taps > 1:
        assert torch.equal(na.conv_state, nb.conv_state)
    for i, (p, q) in enumerate(zip(ga, gb)):
        assert rel_err(p.float(), q.float()) < BF16_TOL, i


# ----------------------------------------------------------------------------------------------
# matrix products of the Linear layers (C ABI: rglru_hip_linear) and the block as one training operator
# ----------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(67, 72, 8), (130, 200, 200), (130, 200, 456), (2050, 2056, 8), (2050, 2056, 200), (2050, 2056, 456)])
def test_forward_product_reads_only_its_operands(M, N, K, dtype):
    """Rows and contraction indices past the operands' edges, which lie inside larger tensors of NaN, leave no trace: one, some and
    many slices of the contraction, none of them a whole number, with small and with large tiles."""
    from griffin_amd import _lib

    lib = _lib.load()
    _say("inside NaN", M, N, K, dtype)
    gen = torch.Generator().manual_seed(11)
    nan = lambda rows, cols: torch.full((rows + 130, cols), float("nan"), dtype=dtype, device="cuda")
    x, w, c = nan(M, K + 64), nan(N, K + 16), nan(M, N + 24)
    x[1:M + 1, 16:16 + K] = torch.randn(M, K, generator=gen).to(dtype).cuda()
    w[1:N + 1, 8:8 + K] = torch.randn(N, K, generator=gen).to(dtype).cuda()
    _lib.check(lib.rglru_hip_linear(0, x[1, 16:].data_ptr(), None, K + 64, w[1, 8:].data_ptr(), None, K + 16, None, None, None, c[1, 8:].data_ptr(),
                                    None, N + 24, None, None, M, N, K, _lib.RGLRU_BF16 if dtype == torch.bfloat16 else _lib.RGLRU_F32,
                                    torch.cuda.current_stream().cuda_stream), "linear")
    torch.cuda.synchronize()
    a, b = x[1:M + 1, 16:16 + K].double(), w[1:N + 1, 8:8 + K].double()
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0         # rounding of the result; then K additions in fp32
    bound = unit * (a @ b.t()).abs() + (K + 2) * 2.0 ** -24 * (a.abs() @ b.abs().t())
    got = c[1:M + 1, 8:8 + N].double()
    assert ((got - a @ b.t()).abs() <= bound).all()
    assert torch.isnan(c[0]).all() and torch.isnan(c[M + 1:]).all() and torch.isnan(c[:, :8]).all() and torch.isnan(c[:, 8 + N:]).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("first", [(0, 1), (3, 2), (5, 0)])
@pytest.mark.parametrize("M,N,K", [(67, 72, 8), (1100, 2056, 72)])
def test_bias_of_a_forward_product_may_start_at_any_element(M, N, K, first, dtype):
    """Biases that are views into longer tensors, on and off the boundaries of the vectors they are loaded as, one of each in a launch;
    what lies around them is NaN.  Small and large tiles, the last of them not full."""
    from griffin_amd import _lib
    from griffin_amd.hip_block_ops import hip_linear

    _say("bias at", first, M, N, K, dtype)
    gen = torch.Generator().manual_seed(first[0])
    make = lambda *shape: torch.randn(*shape, generator=gen).to(dtype).cuda()
    x, weights, biases = make(M, K), [make(N, K) for _ in first], []
    for at in first:
        b = torch.full((at + N + 8,), float("nan"), dtype=dtype, device="cuda")[at:at + N]
        biases.append(b.copy_(make(N)))
        assert b.data_ptr() % 16 == (at * b.element_size()) % 16
    out = [torch.empty(M, N, dtype=dtype, device="cuda") for _ in first]
    _lib.check(_lib.load().rglru_hip_linear(0, x.data_ptr(), None, K, weights[0].data_ptr(), weights[1].data_ptr(), K, biases[0].data_ptr(),
                                            biases[1].data_ptr(), None, out[0].data_ptr(), out[1].data_ptr(), N, None, None, M, N, K,
                                            _lib.RGLRU_BF16 if dtype == torch.bfloat16 else _lib.RGLRU_F32,
                                            torch.cuda.current_stream().cuda_stream), "linear")
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0         # rounding of the result; then K + 1 additions in fp32
    for w, b, got in zip(weights, biases, out):
        want = x.double() @ w.double().t() + b.double()
        bound = unit * want.abs() + (K + 3) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + b.double().abs())
        assert ((got.double() - want).abs() <= bound).all()
        assert torch.equal(hip_linear(x, w, b), got)


# On 256 compute units, small tiles : large: bf16 768 small ones (small), 800 (large); fp32 1024 : 256 (small), 1056 : 264 (small), 2016 : 512
# (large), 2112 : 528 (small)
@pytest.mark.parametrize("dtype,N,M", [(torch.bfloat16, 1024, 3070), (torch.bfloat16, 1024, 3200), (torch.float32, 1024, 4090),
                                       (torch.float32, 1024, 4200), (torch.float32, 2048, 3970), (torch.float32, 2048, 4200)])
@pytest.mark.parametrize("kind,K", [(0, 72), (1, 136)])
def test_linear_products_either_side_of_the_line_between_tiles(kind, K, dtype, N, M):
    """Forward products and input gradients whose rows end inside a tile, on both sides of each line that chooses between small and large
    tiles; what lies behind the operands and around the result is NaN."""
    from griffin_amd import _lib

    _say("tiles", kind, M, N, K, dtype)
    gen = torch.Generator().manual_seed(M)
    nan = lambda rows, cols: torch.full((rows + 130, cols), float("nan"), dtype=dtype, device="cuda")
    a, b, c = nan(M, K), nan(N if kind == 0 else K, K if kind == 0 else N), nan(M, N)
    a[:M] = torch.randn(M, K, generator=gen).to(dtype).cuda()
    b[:-130] = torch.randn(b.size(0) - 130, b.size(1), generator=gen).to(dtype).cuda()
    _lib.check(_lib.load().rglru_hip_linear(kind, a.data_ptr(), None, K, b.data_ptr(), None, b.size(1), None, None, None, c.data_ptr(), None, N, None,
                                            None, M, N, K, _lib.RGLRU_BF16 if dtype == torch.bfloat16 else _lib.RGLRU_F32,
                                            torch.cuda.current_stream().cuda_stream), "linear")
    x, w = a[:M].double(), (b[:N].t() if kind == 0 else b[:K]).double()
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0         # rounding of the result; then K additions in fp32
    bound = unit * (x @ w).abs() + (K + 2) * 2.0 ** -24 * (x.abs() @ w.abs())
    assert ((c[:M].double() - x @ w).abs() <= bound).all() and torch.isnan(c[M:]).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (63, 72, 64), (65, 64, 136), (64, 128, 40), (700, 200, 328), (2050, 2056, 72), (1100, 136, 2304)])
def test_linear_products_match_fp64(M, N, K, dtype):
    """All three kinds at edges of tiles, slices and splits, one and two products a launch, with and without masked rows."""
    from griffin_amd import _lib

    lib = _lib.load()
    code = _lib.RGLRU_BF16 if dtype == torch.bfloat16 else _lib.RGLRU_F32
    _say("products", M, N, K, dtype)
    gen = torch.Generator().manual_seed(7)
    make = lambda *shape: torch.randn(*shape, generator=gen).to(dtype).cuda()
    x, w0, w1, b0, b1 = make(M, K), make(N, K), make(N, K), make(N), make(N)
    dy = make(M, 2 * N)                                          # the halves of one matrix: rows 2 N apart
    keep = torch.rand(M, generator=gen).cuda() < 0.7
    active = keep.to(torch.uint8)
    at = lambda t: None if t is None else t.data_ptr()
    stream = torch.cuda.current_stream().cuda_stream
    tol = 2e-5 if dtype == torch.float32 else 1e-2

    def product(kind, a0, a1, lda, b0_, b1_, ldb, bias0, bias1, act, c0, c1, ldc, partial, sums, m, n, k):
        _lib.check(lib.rglru_hip_linear(kind, at(a0), at(a1), lda, at(b0_), at(b1_), ldb, at(bias0), at(bias1), at(act), at(c0), at(c1), ldc,
                                        at(partial), at(sums), m, n, k, code, stream), "linear")

    def compare(got, want, name):
        torch.cuda.synchronize()
        assert rel_err(got.double().cpu(), want.cpu()) < tol, name

    f = lambda t: t.double()
    y0, y1 = make(M, N), make(M, N)
    product(0, x, None, K, w0, w1, K, b0, b1, active, y0, y1, N, None, None, M, N, K)
    compare(y0, (f(x) @ f(w0).t() + f(b0)) * keep[:, None], "first of two")
    compare(y1, (f(x) @ f(w1).t() + f(b1)) * keep[:, None], "second of two")
    product(0, x, None, K, w0, None, K, None, None, None, y0, None, N, None, None, M, N, K)
    compare(y0, f(x) @ f(w0).t(), "one, no bias")
    dx = make(M, K)
    product(1, dy, dy[:, N:], 2 * N, w0, w1, K, None, None, active, dx, None, K, None, None, M, K, N)
    compare(dx, (f(dy) @ torch.cat((f(w0), f(w1)))) * keep[:, None], "input gradient of two")
    for pair in (1, 2):
        splits = lib.rglru_hip_linear_splits(2, N, K, M, pair, code)
        dw = torch.full((splits, pair, N, K), float("nan"), device="cuda", dtype=torch.float32 if splits > 1 else dtype)
        sums = torch.full((splits, pair, N), float("nan"), device="cuda")
        product(2, dy, dy[:, N:] if pair == 2 else None, 2 * N, x, None, K, None, None, active, dw[0, 0], dw[0, 1] if pair == 2 else None, K,
                dw if splits > 1 else None, sums, N, K, M)
        live = f(dy)[:, :pair * N] * keep[:, None]
        compare(dw.double().sum(0).view(pair * N, K), live.t() @ f(x), "weight gradient")
        compare(sums.double().sum(0).view(-1), live.sum(0), "column sums")


# On 256 compute units, tiles of 64, 128 and 256: input gradients of one and two segments, weight gradients whole and split (the last split
# short); no edge is a whole tile, slice or vector of them
@pytest.mark.parametrize("kind,pair,M,N,K", [(1, 1, 700, 1016, 776), (1, 2, 8200, 776, 1000), (1, 1, 16300, 1016, 776), (1, 2, 33000, 1016, 200),
                                             (2, 1, 1016, 776, 130), (2, 2, 1016, 776, 2331), (2, 1, 776, 1016, 9001), (2, 2, 1016, 776, 16381), (2, 2, 264, 136, 20007)])
@pytest.mark.parametrize("masked", [False, True])
def test_gradient_products_in_every_tile_read_only_their_operands(kind, pair, M, N, K, masked):
    """bf16 gradients against fp64, with operands inside larger tensors of NaN; column sums and masked rows."""
    from griffin_amd import _lib

    lib = _lib.load()
    _say("gradient products", kind, pair, M, N, K, masked)
    gen = torch.Generator(device="cuda").manual_seed(M + K)
    rows_a, cols_a = (M, K) if kind == 1 else (K, M)
    a = torch.full((rows_a + 2, 2 * cols_a + 16), float("nan"), dtype=torch.bfloat16, device="cuda")
    b = torch.full((pair if kind == 1 else 1, K + 2, N + 24), float("nan"), dtype=torch.bfloat16, device="cuda")
    a[1:-1, 8:-8] = torch.randn(rows_a, 2 * cols_a, generator=gen, device="cuda")
    b[:, 1:-1, 8:-16] = torch.randn(b.size(0), K, N, generator=gen, device="cuda")
    if pair == 1:
        a[1:-1, 8 + cols_a:] = float("nan")
    keep = torch.rand(rows_a, generator=gen, device="cuda") < 0.6 if masked else torch.ones(rows_a, dtype=torch.bool, device="cuda")
    active = keep.to(torch.uint8) if masked else None
    at = lambda t: None if t is None else t.data_ptr()
    first, second = a[1, 8:], a[1, 8 + cols_a:] if pair == 2 else None
    ld = a.size(1)
    stream = torch.cuda.current_stream().cuda_stream
    halves = [a[1:-1, 8 + i * cols_a:8 + (i + 1) * cols_a].double() for i in range(pair)]
    if kind == 1:
        c = torch.full((M + 2, N + 24), float("nan"), dtype=torch.bfloat16, device="cuda")
        _lib.check(lib.rglru_hip_linear(1, at(first), at(second), ld, at(b[0, 1, 8:]), at(b[1, 1, 8:]) if pair == 2 else None, b.size(2), None, None,
                                        at(active), at(c[1, 8:]), None, c.size(1), None, None, M, N, K, _lib.RGLRU_BF16, stream), "linear")
        torch.cuda.synchronize()
        want = sum(h @ b[i, 1:-1, 8:-16].double() for i, h in enumerate(halves)) * keep[:, None]
        size = sum(h.abs() @ b[i, 1:-1, 8:-16].double().abs() for i, h in enumerate(halves))
        got = c[1:-1, 8:-16].double()
        # rounding of the result, then 2 K additions in fp32
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + (pair * K + 2) * 2.0 ** -24 * size).all()
        assert torch.isnan(c[0]).all() and torch.isnan(c[-1]).all() and torch.isnan(c[:, :8]).all() and torch.isnan(c[:, -16:]).all()
        return
    splits = lib.rglru_hip_linear_splits(2, M, N, K, pair, _lib.RGLRU_BF16)
    dw = torch.full((splits, pair, M, N), float("nan"), device="cuda", dtype=torch.float32 if splits > 1 else torch.bfloat16)
    sums = torch.full((splits, pair, M), float("nan"), device="cuda")
    _lib.check(lib.rglru_hip_linear(2, at(first), at(second), ld, at(b[0, 1, 8:]), None, b.size(2), None, None, at(active), at(dw[0, 0]),
                                    at(dw[0, 1]) if pair == 2 else None, N, at(dw) if splits > 1 else None, at(sums), M, N, K, _lib.RGLRU_BF16, stream), "linear")
    torch.cuda.synchronize()
    x = b[0, 1:-1, 8:-16].double()
    for i, h in enumerate(halves):
        live = h * keep[:, None]
        want, size = live.t() @ x, live.abs().t() @ x.abs()
        unit = 2.0 ** -8 if splits == 1 else 0.0
        assert ((dw.double().sum(0)[i] - want).abs() <= unit * want.abs() + (K + 2) * 2.0 ** -24 * size).all()
        assert ((sums.double().sum(0)[i] - live.sum(0)).abs() <= (K + 2) * 2.0 ** -24 * live.abs().sum(0)).all()


# multiply-adds between the lines of inference and of gradients, and past both with tokens that do not divide into 2048
@pytest.mark.parametrize("rows,N,K", [(1100, 2048, 2816), (2200, 2048, 2816)])
def test_linear_layers_take_batches_of_gradients(rows, N, K):
    """Batched gradients have no memory for a kernel to read: hip_linear and hip_linear_pair give them to PyTorch's products, one by one the same."""
    from griffin_amd.hip_block_ops import hip_linear, hip_linear_pair

    _say("batched gradients", rows, N, K)
    gen = torch.Generator(device="cuda").manual_seed(3)
    x, w1, w2 = (torch.randn(*s, generator=gen, device="cuda").bfloat16().requires_grad_(True) for s in ((rows, K), (N, K), (N, K)))
    dy = torch.randn(2, 2, rows, N, generator=gen, device="cuda").bfloat16()
    for outs, leaves in (([hip_linear(x, w1, None)], (x, w1)), (list(hip_linear_pair(x, w1, None, w2, None)), (x, w1, w2))):
        both = torch.autograd.grad(outs, leaves, [dy[i] for i in range(len(outs))], retain_graph=True, is_grads_batched=True)
        for i in range(2):
            for got, want in zip(both, torch.autograd.grad(outs, leaves, [dy[j, i] for j in range(len(outs))], retain_graph=True)):
                assert rel_err(got[i].float(), want.float()) < 1e-2      # two roundings to bf16, sums in another order


@pytest.mark.parametrize("padded", [False, True])
@pytest.mark.parametrize("B,T,D,W,nb", [(2, 1, 64, 96, 3), (3, 37, 72, 128, 2), (2, 333, 192, 256, 16), (2, 4097, 768, 1024, 16), (4, 2048, 1536, 2048, 16)])
def test_block_as_one_training_operator_matches_layer_by_layer(B, T, D, W, nb, padded):
    """The node that covers the whole block (own products and, for the long ones, those of the BLAS library) against the same
    block taken layer by layer, which is what a call that returns a cache does."""
    from griffin_amd import RecurrentBlock

    _say("block as one operator", B, T, D, W, nb, padded)
    torch.manual_seed(5)
    block = RecurrentBlock(D, W, gate_blocks=nb, scan_mode="hip").cuda().to(torch.bfloat16)
    with torch.no_grad():
        for name, p in block.named_parameters():
            if name.endswith("bias"):
                p.normal_(std=0.1)
    x = torch.randn(B, T, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    dy = torch.randn_like(x)
    active = None
    if padded:
        lengths = torch.linspace(max(1, T // 5), T, B, device="cuda").long()
        active = torch.arange(T, device="cuda")[None] < lengths[:, None]
    names, leaves = zip(*([("x", x)] + list(block.named_parameters())))
    nodes = []
    whole = block(x, active_mask=active)
    nodes.append(type(whole.grad_fn).__name__ + str(whole.grad_fn.name()))
    assert "BlockTrain" in nodes[0]
    got = torch.autograd.grad(whole, leaves, dy)
    layered, _ = block(x, active_mask=active, return_cache=True)
    want = torch.autograd.grad(layered, leaves, dy)
    torch.cuda.synchronize()
    assert rel_err(whole.float(), layered.float()) < 1e-2
    for name, g, w in zip(names, got, want):
        err = float((g.float() - w.float()).norm() / w.float().norm().clamp_min(1e-30))
        _say("  d%s rel error: %.2e" % (name, err))
        assert err < 1e-2, name


# multiply-adds of a product: 1.04e10 (gradients by the library, forward by the BLAS library), 2.6e10 with tokens that do not divide into the
# BLAS library's batches (weight gradients by the library alone).  The padded batches are packed to 1984 and 5056 rows: 6.2e9, all products by the
# library, and 1.6e10; padding that stays is the next test's.
@pytest.mark.parametrize("padded", [False, True])
@pytest.mark.parametrize("B,T,D,W,nb", [(3, 1100, 1536, 2048, 16), (3, 2777, 1536, 2048, 16)])
def test_block_training_between_the_lines_of_its_products(B, T, D, W, nb, padded):
    test_block_as_one_training_operator_matches_layer_by_layer(B, T, D, W, nb, padded)


# multiply-adds of a product, tokens: 1.04e10 and 1.03e10 (gradients by the library, forward by the BLAS library), 3300 and 2 x 2048;  2.6e10 and
# 1.3e10 (input gradients by the BLAS library; weight gradients by the library in 8331 tokens, by the BLAS library in 8 x 2048)
@pytest.mark.parametrize("B,T,D,W,nb", [(3, 1100, 1536, 2048, 16), (4, 1024, 1408, 1792, 16), (3, 2777, 1536, 2048, 16), (8, 2048, 768, 1024, 8)])
@pytest.mark.parametrize("how", ["little padding", "positions"])
def test_block_trains_on_long_right_padded_batches_with_their_padding(B, T, D, W, nb, how):
    """Right-padded batches that are not packed, for little padding (90 % active) or because the caller gives positions: the node with masked
    products and row masks against the block taken layer by layer, on either side of the lines of its products."""
    from griffin_amd import RecurrentBlock, hip_block_ops

    _say("padded block, not packed", B, T, D, W, nb, how)
    torch.manual_seed(6)
    block = RecurrentBlock(D, W, gate_blocks=nb, scan_mode="hip").cuda().to(torch.bfloat16)
    with torch.no_grad():
        for name, p in block.named_parameters():
            if name.endswith("bias"):
                p.normal_(std=0.1)
    x = torch.randn(B, T, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    dy = torch.randn_like(x)
    positions = torch.arange(T, device="cuda").repeat(B, 1) if how == "positions" else None
    active = torch.arange(T, device="cuda")[None] < torch.linspace(T // 5 if how == "positions" else 4 * T // 5, T, B, device="cuda").long()[:, None]
    names, leaves = zip(*([("x", x)] + list(block.named_parameters())))
    calls, real = [], hip_block_ops.hip_block_train_packed

    def spy(*args):
        calls.append(real(*args))
        return calls[-1]

    hip_block_ops.hip_block_train_packed = spy
    try:
        whole = block(x, segment_pos=positions, active_mask=active)
    finally:
        hip_block_ops.hip_block_train_packed = real
    assert calls == ([None] if positions is None else []) and "BlockTrain" in type(whole.grad_fn).__name__ + str(whole.grad_fn.name())
    got = torch.autograd.grad(whole, leaves, dy)
    layered, _ = block(x, segment_pos=positions, active_mask=active, return_cache=True)
    want = torch.autograd.grad(layered, leaves, dy)
    torch.cuda.synchronize()
    assert (whole[~active] == 0).all() and (got[0][~active] == 0).all()
    assert rel_err(whole.float(), layered.float()) < 1e-2
    for name, g, w in zip(names, got, want):
        err = float((g.float() - w.float()).norm() / w.float().norm().clamp_min(1e-30))
        _say("  d%s rel error: %.2e" % (name, err))
        assert err < 1e-2, name


@pytest.mark.parametrize("B,T,counts,packed", [(1, 1, [1], 1), (3, 16, [16, 0, 5], 64), (5, 37, [1, 0, 37, 17, 16], 71), (300, 70, None, 11520), (2, 5000, [4999, 3], 5056),
                                               (2, 3, [1, 2], 700)])
def test_rows_are_packed_and_unpacked(B, T, counts, packed):
    """Rows without their padding and back, for counts at the edges of a workgroup's tokens, empty rows, and a rest longer than a row: two
    arrays of different widths, positions and flags; nothing outside the results is written."""
    from griffin_amd import _lib

    lib = _lib.load()
    _say("pack", B, T, packed)
    gen = torch.Generator().manual_seed(T)
    if counts is None:
        counts = torch.randint(0, T + 1, (B,), generator=gen).tolist()
    assert sum(counts) <= packed
    stream = torch.cuda.current_stream().cuda_stream
    device = torch.tensor(counts, dtype=torch.int32, device="cuda")
    live = torch.arange(T)[None] < torch.tensor(counts)[:, None]
    wide = [torch.randn(B, T, n, generator=gen).cuda() for n in (4, 92)]
    narrow = [torch.full((packed + 1, n), 7.0, device="cuda") for n in (4, 92)]
    pos, flags = torch.full((packed + 1,), -7, device="cuda"), torch.full((packed + 1,), 77, dtype=torch.uint8, device="cuda")
    _lib.check(lib.rglru_hip_pack_rows(device.data_ptr(), wide[0].data_ptr(), narrow[0].data_ptr(), 16, wide[1].data_ptr(), narrow[1].data_ptr(), 368,
                                       pos.data_ptr(), flags.data_ptr(), B, T, packed, stream), "pack_rows")
    rest = packed - sum(counts)
    for x, y in zip(wide, narrow):
        want = torch.cat((x.cpu()[live], torch.zeros(rest, x.size(2)), torch.full((1, x.size(2)), 7.0)))
        assert torch.equal(y.cpu(), want)
        back = torch.full((B * T + 1, x.size(2)), 7.0, device="cuda")
        _lib.check(lib.rglru_hip_unpack_rows(device.data_ptr(), y.data_ptr(), back.data_ptr(), 4 * x.size(2), B, T, packed, stream), "unpack_rows")
        assert torch.equal(back[:-1].cpu().view(B, T, -1), x.cpu() * live[:, :, None]) and (back[-1] == 7.0).all()
    want = torch.cat([torch.arange(n) for n in (*counts, rest)])
    assert torch.equal(pos.cpu(), torch.cat((want, torch.tensor([-7]))))
    near = (3 - want.clamp(max=3)) << 2                          # RGLRU_FLAG_CONV_SHIFT
    assert torch.equal(flags.cpu(), torch.cat(((near | (want == 0)), torch.tensor([77]))).to(torch.uint8))


def test_rows_past_the_packed_ones_are_not_touched():
    """Counts that say more than there is: a row has at most T tokens, and what does not fit the packed rows is dropped by either direction (every array
    here has memory behind its end)."""
    from griffin_amd import _lib

    _say("pack", "counts that do not fit")
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    B, T, packed = 2, 5, 8
    counts = torch.tensor([4, 9], dtype=torch.int32, device="cuda")                      # 4 and T; 8 of the 9 rows fit
    wide = torch.full((B * T + 8, 4), float("nan"), device="cuda")
    wide[:B * T] = torch.arange(1.0, B * T + 1)[:, None]
    narrow, back = torch.full((packed + 8, 4), 7.0, device="cuda"), torch.full((B * T + 8, 4), 7.0, device="cuda")
    _lib.check(lib.rglru_hip_pack_rows(counts.data_ptr(), wide.data_ptr(), narrow.data_ptr(), 16, None, None, 0, None, None, B, T, packed, stream), "pack_rows")
    narrow[packed:] = float("nan")
    _lib.check(lib.rglru_hip_unpack_rows(counts.data_ptr(), narrow.data_ptr(), back.data_ptr(), 16, B, T, packed, stream), "unpack_rows")
    assert narrow[:, 0].tolist()[:packed] == [1, 2, 3, 4, 6, 7, 8, 9]
    assert back[:, 0].tolist() == [1, 2, 3, 4, 0, 6, 7, 8, 9, 0] + [7] * 8


@pytest.mark.parametrize("B,T,D,W,nb,lengths", [(5, 1700, 768, 1024, 8, [0, 1, 2, 3, 1700]), (150, 33, 768, 1024, 16, None), (3, 2000, 640, 832, 8, [2000, 1, 1500]),
                                                (9, 2048, 768, 1024, 16, [2048, 2048, 5, 2048, 64, 128, 2047, 1, 513]), (4, 1100, 768, 1024, 8, [0, 0, 0, 0])])
def test_block_trains_on_right_padded_batches_without_their_padding(B, T, D, W, nb, lengths):
    """Long right-padded batches run on their active tokens alone: output and gradients against the block taken layer by layer, whatever
    lies in the padding; a second backward pass over the same forward repeats."""
    from griffin_amd import RecurrentBlock, hip_block_ops

    _say("packed block", B, T, D, W, nb)
    torch.manual_seed(5)
    lengths = torch.tensor(lengths if lengths is not None else [(7 * i) % (T + 1) for i in range(B)])
    block = RecurrentBlock(D, W, gate_blocks=nb, scan_mode="hip").cuda().to(torch.bfloat16)
    with torch.no_grad():
        for name, p in block.named_parameters():
            if name.endswith("bias"):
                p.normal_(std=0.1)
    active = (torch.arange(T)[None] < lengths[:, None]).cuda()
    x = torch.randn(B, T, D, device="cuda", dtype=torch.bfloat16)
    dy = torch.randn_like(x)
    names, leaves = zip(*block.named_parameters())
    calls, real = [], hip_block_ops.hip_block_train_packed

    def spy(*args):
        calls.append(real(*args))
        return calls[-1]

    hip_block_ops.hip_block_train_packed = spy
    try:
        dirty = x.masked_fill(~active[:, :, None], float("nan")).requires_grad_(True)
        whole = block(dirty, active_mask=active)
    finally:
        hip_block_ops.hip_block_train_packed = real
    assert len(calls) == 1 and calls[0] is not None
    got = torch.autograd.grad(whole, (dirty, *leaves), dy.masked_fill(~active[:, :, None], float("nan")), retain_graph=True)
    again = torch.autograd.grad(whole, (dirty, *leaves), dy)
    x.requires_grad_(True)
    layered, _ = block(x, active_mask=active, return_cache=True)
    want = torch.autograd.grad(layered, (x, *leaves), dy)
    torch.cuda.synchronize()
    assert (whole[~active] == 0).all() and (got[0][~active] == 0).all()
    assert rel_err(whole.float(), layered.float()) < 1e-2
    for name, g, a, w in zip(("x", *names), got, again, want):
        norm = w.float().norm().clamp_min(1e-30)
        err = float((g.float() - w.float()).norm() / norm)
        _say("  d%s rel error: %.2e" % (name, err))
        assert err < 1e-2 and float((a.float() - w.float()).norm() / norm) < 1e-2, name


# multiply-adds of a projection: 3.1e9, 7.1e9, 1.3e10
@pytest.mark.parametrize("B,T,together", [(4, 1000, True), (8, 1125, True), (8, 2048, False)])
def test_projections_of_a_batch_that_may_be_packed_are_one_launch_where_they_can(B, T, together):
    """Both projections are queued in front of the wait for the mask where they are one launch, and an all-true mask then asks for no other; the
    values are those of the two layers."""
    from griffin_amd import RecurrentBlock, hip_block_ops

    _say("projections in front of the mask", B, T)
    torch.manual_seed(2)
    block = RecurrentBlock(768, 1024, gate_blocks=16, scan_mode="hip").cuda().to(torch.bfloat16)
    x = torch.randn(B, T, 768, device="cuda", dtype=torch.bfloat16)
    layers = block.linear_x, block.linear_y
    assert hip_block_ops.hip_block_may_pack(x, layers[0].weight)
    u, v = hip_block_ops.hip_block_projections(x, *(t for m in layers for t in (m.weight, m.bias)))
    assert (v is not None) == together
    for got, m in zip((u, v), layers):
        if got is not None:
            assert rel_err(got.float(), torch.nn.functional.linear(x.float(), m.weight.float(), m.bias.float())) < 4e-3      # one rounding to bf16
    alone, real = [], hip_block_ops.hip_linear_values
    hip_block_ops.hip_linear_values = lambda *args: alone.append(1) or real(*args)
    try:
        block(x.requires_grad_(True), active_mask=torch.ones(B, T, dtype=torch.bool, device="cuda"))
    finally:
        hip_block_ops.hip_linear_values = real
    assert len(alone) == (0 if together else 1)


@pytest.mark.parametrize("tokens", ["all", "positions", "padded"])
@pytest.mark.parametrize("B,T,D,W,nb,carried", [(2, 2, 64, 96, 3, True), (3, 77, 72, 128, 2, True), (1, 1000, 192, 256, 16, False), (3, 2777, 1536, 2048, 16, True)])
def test_block_inference_in_one_call_matches_layer_by_layer(B, T, D, W, nb, carried, tokens):
    """Output and cache of the inference call that covers the whole block against the same block with one launch per layer
    (a forward hook on a layer takes it there)."""
    from griffin_amd import RecurrentBlock, RecurrentBlockCache, hip_block_ops

    _say("block inference", B, T, D, W, nb, carried, tokens)
    torch.manual_seed(6)
    block = RecurrentBlock(D, W, gate_blocks=nb, scan_mode="hip").cuda().to(torch.bfloat16).eval()
    x = torch.randn(B, T, D, device="cuda", dtype=torch.bfloat16)
    cache = None
    if carried:
        cache = RecurrentBlockCache(torch.randn(B, W, device="cuda"), torch.randn(B, 3, W, device="cuda", dtype=torch.bfloat16),
                                    torch.tensor([99, 0, -1][:B], device="cuda"))
    kwargs = {}
    if tokens == "positions":
        position = torch.arange(T, device="cuda").repeat(B, 1)
        position[:, T // 2:] -= T // 2
        kwargs["segment_pos"] = position
    elif tokens == "padded":
        lengths = torch.linspace(max(1, T // 5), T, B, device="cuda").long()
        kwargs["active_mask"] = torch.arange(T, device="cuda")[None] < lengths[:, None]
    calls, real = [], hip_block_ops.hip_block_infer
    hip_block_ops.hip_block_infer = lambda *args: calls.append(1) or real(*args)
    try:
        with torch.no_grad():
            got, got_cache = block(x, cache, return_cache=True, **kwargs)
            assert calls
            handle = block.temporal_conv.register_forward_hook(lambda *args: None)
            want, want_cache = block(x, cache, return_cache=True, **kwargs)
            handle.remove()
    finally:
        hip_block_ops.hip_block_infer = real
    torch.cuda.synchronize()
    assert len(calls) == 1
    assert rel_err(got.float(), want.float()) < 1e-2
    assert rel_err(got_cache.rnn_state, want_cache.rnn_state) < 1e-2
    assert torch.equal(got_cache.segment_position, want_cache.segment_position)
    assert rel_err(got_cache.conv_state.float(), want_cache.conv_state.float()) < 1e-2


# one tile and the smallest width; rows that end inside tiles of 64; tiles of 128
@pytest.mark.parametrize("B,T,D,W,nb", [(1, 1, 8, 96, 3), (9, 77, 72, 128, 2), (3, 1537, 136, 2048, 16)])
@pytest.mark.parametrize("tokens", ["fresh", "continued", "positions"])
def test_projections_carry_the_positions_of_an_inference_call(B, T, D, W, nb, tokens):
    """rglru_hip_block_project: flag bytes and last positions for every kind of position, the products of rglru_hip_linear bit for bit, and a
    workspace that held anything is cleared for the forward behind it."""
    from griffin_amd import _lib

    _say("projections with positions", B, T, D, W, nb, tokens)
    lib, code = _lib.load(), _lib.RGLRU_BF16
    gen = torch.Generator().manual_seed(11)
    make = lambda *shape: torch.randn(*shape, generator=gen).to(torch.bfloat16).cuda()
    x, w0, w1, b0, b1 = make(B, T, D), make(W, D), make(W, D), make(W), make(W)
    prev = torch.tensor([-1, 0, 1, 2, 3, 2 ** 40, -2, -3, -2 ** 40])[:B].cuda() if tokens == "continued" else None
    seg = torch.randint(-3, 6, (B, T), generator=gen).cuda() if tokens == "positions" else None
    pos = seg if seg is not None else (prev[:, None] + 1 if prev is not None else 0) + torch.arange(T, device="cuda").repeat(B, 1)
    bytes_ = lambda n: torch.full((n,), 0xff, dtype=torch.uint8, device="cuda")
    ws, flags = bytes_(lib.rglru_hip_workspace_bytes(B, T, W, nb)), bytes_(B * T + 8)
    last = torch.full((B + 1,), -7, device="cuda")
    u, v, u2, v2 = (torch.full((B * T + 1, W), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(4))
    at = lambda t: None if t is None else t.data_ptr()
    stream = torch.cuda.current_stream().cuda_stream
    held = None if tokens == "fresh" else at(flags)
    _lib.check(lib.rglru_hip_block_project(at(x), at(w0), at(w1), at(b0), at(b1), at(u), at(v), at(prev), at(seg), held, at(last), at(ws), B, T, D,
                                           W, nb, code, stream), "project")
    _lib.check(lib.rglru_hip_linear(0, at(x), None, D, at(w0), at(w1), D, at(b0), at(b1), None, at(u2), at(v2), W, None, None, B * T, W, D, code,
                                    stream), "linear")
    torch.cuda.synchronize()
    for got, want in ((u, u2), (v, v2)):
        assert torch.equal(got[:-1], want[:-1]) and torch.isnan(got[-1]).all()
    want = (pos == 0).to(torch.uint8) | ((3 - pos).clamp(0, 3) << 2).to(torch.uint8)
    assert torch.equal(flags[:B * T].view(B, T), want) if held else (flags == 0xff).all()
    assert (flags[B * T:] == 0xff).all() and torch.equal(last[:-1], pos[:, -1]) and int(last[-1]) == -7
    # the forward behind it, against the one that launches its own positions
    gates = [make(nb, W // nb, W // nb) * 0.1, make(nb, W // nb) * 0.1, make(nb, W // nb, W // nb) * 0.1, make(nb, W // nb) * 0.1]
    a_param = torch.rand(W, generator=gen).to(torch.bfloat16).cuda()
    prep = bytes_(lib.rglru_hip_prep_bytes(W, nb, code))
    _lib.check(lib.rglru_hip_prepare(*(at(t) for t in gates), at(a_param), 8.0, W, nb, code, code, at(prep), stream), "prepare")
    taps, bias, state, h0 = make(W, 4), make(W), make(B, 3, W), torch.randn(B, W, generator=gen).cuda()
    results = []
    for own in (True, False):
        gated, new_state, h = (torch.full(s, float("nan"), dtype=t, device="cuda") for s, t in
                               (((B, T, W), torch.bfloat16), ((B, 3, W), torch.bfloat16), ((B, W), torch.float32)))
        common = (at(u), W, at(v), W, at(state), at(taps), at(bias), 4, code, at(prep), at(h0))
        if own:
            _lib.check(lib.rglru_hip_block_infer_projected(*common, held, at(gated), at(new_state), at(h), at(ws), B, T, W, nb, code, stream), "behind")
        else:
            again = bytes_(B * T)
            _lib.check(lib.rglru_hip_block_infer(*common, at(prev), at(seg), at(again) if held else None, at(gated), at(new_state), at(h), at(last),
                                                 at(ws), B, T, W, nb, code, stream), "infer")
        torch.cuda.synchronize()
        results.append((gated, new_state, h))
    for got, want in zip(*results):
        assert rel_err(got.float(), want.float()) < 4e-3      # one rounding to bf16; the order in which tiles pass the state may differ
    # refused: no workspace, no place for the flags
    refused = lambda *edit: lib.rglru_hip_block_project(at(x), at(w0), at(w1), at(b0), at(b1), at(u), at(v), None, *edit, B, T, D, W, nb, code, stream)
    assert refused(None, None, at(last), None) != 0 and refused(at(pos.contiguous()), None, at(last), at(ws)) != 0


# On 256 compute units, tiles of 64 x 64, 128 x 64, 128 x 128 and 192 x 128; no edge is a whole tile or slice of them
@pytest.mark.parametrize("pair,M,N,K", [(1, 700, 1016, 776), (2, 777, 1016, 776), (1, 2331, 776, 1000), (2, 2331, 1016, 776), (1, 8200, 1016, 776), (2, 6000, 1000, 264), (2, 14000, 1016, 72)])
@pytest.mark.parametrize("masked", [False, True])
def test_forward_products_in_every_tile_read_only_their_operands(pair, M, N, K, masked):
    """bf16 forward products against fp64, with operands inside larger tensors of NaN; biases on and off the boundaries of vectors; masked rows."""
    from griffin_amd import _lib

    _say("forward products", pair, M, N, K, masked)
    gen = torch.Generator(device="cuda").manual_seed(M + K)
    nan = lambda *shape: torch.full(shape, float("nan"), dtype=torch.bfloat16, device="cuda")
    x, w, c, bias = nan(M + 2, K + 24), nan(pair, N + 2, K + 16), nan(pair, M + 2, N + 24), nan(pair, N + 11)
    x[1:-1, 8:-16] = torch.randn(M, K, generator=gen, device="cuda")
    w[:, 1:-1, 8:-8] = torch.randn(pair, N, K, generator=gen, device="cuda")
    starts = (8, 3)
    for i in range(pair):
        bias[i, starts[i]:starts[i] + N] = torch.randn(N, generator=gen, device="cuda")
    keep = torch.rand(M, generator=gen, device="cuda") < 0.6 if masked else torch.ones(M, dtype=torch.bool, device="cuda")
    active = keep.to(torch.uint8) if masked else None
    at = lambda t: None if t is None else t.data_ptr()
    second = lambda t: at(t) if pair == 2 else None
    _lib.check(_lib.load().rglru_hip_linear(0, at(x[1, 8:]), None, x.size(1), at(w[0, 1, 8:]), second(w[-1, 1, 8:]), w.size(2), at(bias[0, 8:]), second(bias[-1, 3:]),
                                            at(active), at(c[0, 1, 8:]), second(c[-1, 1, 8:]), c.size(2), None, None, M, N, K, _lib.RGLRU_BF16,
                                            torch.cuda.current_stream().cuda_stream), "linear")
    torch.cuda.synchronize()
    xs = x[1:-1, 8:-16].double()
    for i in range(pair):
        ws, b = w[i, 1:-1, 8:-8].double(), bias[i, starts[i]:starts[i] + N].double()
        want = (xs @ ws.t() + b) * keep[:, None]
        size = xs.abs() @ ws.abs().t() + b.abs()
        got = c[i, 1:-1, 8:-16].double()
        # rounding of the result, then K additions in fp32
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + (K + 2) * 2.0 ** -24 * size).all()
        assert torch.isnan(c[i, 0]).all() and torch.isnan(c[i, -1]).all() and torch.isnan(c[i, :, :8]).all() and torch.isnan(c[i, :, -16:]).all()

"""One decoded token of a GDN block in three launches (gdn_decode.hip), against the float64 block oracle's steps and
against the step-by-step path, where its kernels can go wrong: one to 17 sequences (the projections' kernel takes 8 at a
time, up to 16), odd row counts and input widths, one, two and four value heads per key head, empty and full caches, each dtype."""

import numpy as np
import pytest
import torch

from oracle import gdn_oracle as O

pytestmark = pytest.mark.gpu

D = 128


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gdn_lib
    gdn_lib.load()
    return torch.device("cuda:0")


@pytest.mark.parametrize("dtype,tokens,k,rows", [
    (torch.float32, 1, 8, (1, 5, 64, 3)), (torch.bfloat16, 2, 520, (257, 4)), (torch.bfloat16, 3, 2048, (33,)),
    (torch.float16, 5, 1000, (7, 130)), (torch.bfloat16, 8, 4096, (64, 9, 8)), (torch.bfloat16, 13, 256, (33, 5))])
def test_small_linears(dev, dtype, tokens, k, rows):
    import gdn_block
    gen = torch.Generator(device=dev).manual_seed(k)
    n = lambda *s: torch.randn(*s, device=dev, generator=gen).to(dtype)
    x, ws = n(tokens, k), [n(r, k) for r in rows]
    # sums of k products in fp32 (k 2^-24 of their absolute sum), then one rounding to the dtype
    eps = torch.finfo(dtype).eps
    for y, w in zip(gdn_block.small_linears(x, ws), ws):
        ref = x.double() @ w.double().t()
        bar = eps * ref.abs() + k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
        assert bool(((y.double() - ref).abs() <= bar).all())


def _token64(blk, x, conv, state):
    """The block's steps for one token in float64 (oracle functions)."""
    W = lambda m: getattr(blk, m).weight.detach().double().cpu().numpy()
    qkv, z, b, a = (x @ W(m).T for m in ("in_proj_qkv", "in_proj_z", "in_proj_b", "in_proj_a"))
    B, Hk, Hv = x.shape[0], blk.Hk, blk.Hv
    seq = np.concatenate([conv, qkv[:, None]], 1)
    c = O.silu((seq * W("conv1d")[:, 0].T[None]).sum(1))
    kd = Hk * D
    q, k, v = c[:, :kd].reshape(B, Hk, D), c[:, kd:2 * kd].reshape(B, Hk, D), c[:, 2 * kd:].reshape(B, Hv, D)
    q, k = O.l2norm(q, 1e-6, D ** -0.5), O.l2norm(k, 1e-6, 1.0)
    dec, beta = O.gates(a, b, blk.A_log.detach().double().cpu().numpy(), blk.dt_bias.detach().double().cpu().numpy())
    q, k = np.repeat(q, Hv // Hk, 1), np.repeat(k, Hv // Hk, 1)
    A = state * dec[..., None, None]
    delta = beta[..., None] * (v - (A * k[:, :, None]).sum(-1))
    S = A + delta[..., None] * k[:, :, None]
    y = (S * q[:, :, None]).sum(-1)
    zh = z.reshape(B, Hv, D)
    o = y / np.sqrt((y * y).mean(-1, keepdims=True) + blk.norm.eps) * W("norm") * O.silu(zh)
    return o.reshape(B, -1) @ W("out_proj").T, seq[:, 1:], S


@pytest.mark.parametrize("dtype,B,Hk,Hv,hidden,empty", [
    (torch.float32, 1, 2, 4, 72, False), (torch.bfloat16, 3, 1, 4, 264, False), (torch.bfloat16, 9, 2, 2, 256, False),
    (torch.bfloat16, 17, 1, 2, 128, False),
    (torch.float16, 8, 2, 4, 100, False), (torch.bfloat16, 1, 2, 4, 256, True)])
def test_block_token(dev, dtype, B, Hk, Hv, hidden, empty):
    import qwen3_5 as Q
    torch.manual_seed(B)
    blk = Q.GatedDeltaNet(Q.ModelArgs(hidden_size=hidden, linear_num_key_heads=Hk, linear_num_value_heads=Hv,
                                      linear_key_head_dim=D, linear_value_head_dim=D)).to(dev, dtype).eval()
    x = torch.randn(B, 1, hidden, device=dev).to(dtype)
    conv, state = torch.randn(B, 3, blk.conv_dim, device=dev), 0.1 * torch.randn(B, Hv, D, D, device=dev)
    caches = [Q.GDNCache(), Q.GDNCache()]
    if not empty:
        for c in caches:
            c[0], c[1] = conv, state
    with torch.no_grad():
        assert blk._decodes_fused(x, caches[0])
        fused = [blk(x, cache=caches[0]), caches[0][0], caches[0][1]]
        hook = blk.norm.register_forward_hook(lambda *a: None)  # a hooked block runs step by step
        assert not blk._decodes_fused(x, caches[1])
        steps = [blk(x, cache=caches[1]), caches[1][0], caches[1][1]]
        hook.remove()
    z = 0.0 if empty else 1.0
    want = _token64(blk, x[:, 0].double().cpu().numpy(), z * conv.double().cpu().numpy(), z * state.double().cpu().numpy())
    # a few roundings to the dtype in a row (the step-by-step path has more of them); fp32: sums and exp
    bar = {torch.float32: 1e-5, torch.float16: 4e-3, torch.bfloat16: 3e-2}[dtype]
    for name, f, s, w in zip(("out", "conv", "state"), fused, steps, want):
        f, s = (t.double().cpu().numpy().reshape(w.shape) for t in (f, s))
        scale = np.abs(w).max()
        assert np.abs(f - w).max() <= bar * scale, name
        assert np.abs(f - s).max() <= 2 * bar * scale, name


def test_calls_that_run_step_by_step(dev):
    """Training, gradients, autocast, biases, a replaced update and caches of another layout keep the general path."""
    import qwen3_5 as Q
    blk = Q.GatedDeltaNet(Q.ModelArgs(hidden_size=64, linear_num_key_heads=1, linear_num_value_heads=2,
                                      linear_key_head_dim=D, linear_value_head_dim=D)).to(dev).eval()
    x, c = torch.randn(2, 1, 64, device=dev), Q.GDNCache()
    assert blk._decodes_fused(x, c)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not blk._decodes_fused(x, c)
    assert not blk.train()._decodes_fused(x, c)
    blk.eval()
    c[1] = torch.zeros(2, D, 2, D, device=dev).transpose(1, 2)
    assert not blk._decodes_fused(x, c)
    c[1] = torch.zeros(2, 2, D, D, device=dev, dtype=torch.float64)
    assert not blk._decodes_fused(x, c)
    c[1] = None
    keep, Q.gated_delta_update = Q.gated_delta_update, lambda *a, **k: keep(*a, **k)
    try:
        assert not blk._decodes_fused(x, c)
    finally:
        Q.gated_delta_update = keep
    blk.out_proj = torch.nn.Linear(2 * D, 64, bias=True, device=dev)
    assert not blk._decodes_fused(x, c)


def test_unknown_form_is_refused(dev, monkeypatch):
    """GDN_FORM names no form: the fused token raises what the step-by-step one does, and leaves the cache alone."""
    import qwen3_5 as Q
    blk = Q.GatedDeltaNet(Q.ModelArgs(hidden_size=64, linear_num_key_heads=1, linear_num_value_heads=2,
                                      linear_key_head_dim=D, linear_value_head_dim=D)).to(dev).eval()
    x, c = torch.randn(2, 1, 64, device=dev), Q.GDNCache()
    monkeypatch.setenv("GDN_FORM", "chunked")
    with torch.no_grad(), pytest.raises(ValueError, match="GDN_FORM"):
        blk(x, cache=c)
    assert c[0] is None and c[1] is None

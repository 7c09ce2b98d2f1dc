"""The low halves of a masked bf16 call.  Its query rows q~ = d (q - beta c k), the chunk-entry states and an fp32 dy are
bf16 values plus what those leave (hi and lo), and every result that has no other rounding to 16 bits has to keep both:
y, dg, dbeta, dS0, and dq and dk as the C ABI gives them in fp32.  Against the fp64 oracle on calls where nothing else is
rounded: one unmasked token, then masked ones, so that no W h, no M and no second chunk's Delta enters."""

import numpy as np
import pytest
import torch

from oracle import gdn_oracle as O

pytestmark = pytest.mark.gpu

D = 128
# A hi / lo pair leaves 2^-18 of a value, the product of two lo halves is dropped (2^-18), and three pairs meet at most
# (q~, P or dP, and the state or Delta): 2^-16 of the norm, with a factor of 4 for sums that cancel in part.  Without one
# of the lo halves the error is the rounding to 8 bits, 2^-9.3 of the norm (rms).
BAR = 2.0 ** -14


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gdn_lib
    gdn_lib.load()
    return torch.device("cuda:0")


def _call(d, dev, chunk, dy_dtype):
    """gdn_fwd and gdn_bwd with y and every gradient in fp32."""
    import gdn_lib as L
    lib = L.load()
    t = lambda x, dt=torch.float32: torch.tensor(x, device=dev).to(dt).contiguous()
    q, k, v = (t(d[n], torch.bfloat16) for n in "qkv")
    g, beta, state, dy = t(d["decay"]), t(d["beta"]), t(d["state"]), t(d["dy"], dy_dtype)
    mask = t(d["mask"], torch.uint8)
    (B, T, Hk, _), Hv = q.shape, v.shape[2]
    shape, st = (B, T, Hk, Hv, D, D, chunk), L.stream_handle(dev)
    gate, form, code = L.GATE_DECAY, L.FORM_CHUNK, L.BF16
    new = lambda *s, dt=torch.float32: torch.empty(s, device=dev, dtype=dt)
    saved = new(lib.gdn_saved_bytes(*shape, gate, 1, form, code), dt=torch.uint8)
    ws = new(max(1, lib.gdn_fwd_workspace_bytes(*shape, gate, 1, form, code, 1)), dt=torch.uint8)
    y, S = new(B, T, Hv, D), new(B, Hv, D, D)
    p = L.ptr
    L.check(lib.gdn_fwd(p(q), p(k), p(v), p(g), p(beta), p(state), p(mask), p(y), p(S), p(saved), saved.numel(), p(ws),
                        ws.numel(), *shape, code, L.F32, gate, form, st))
    wb = new(lib.gdn_bwd_workspace_bytes(*shape, gate, 1, form, code), dt=torch.uint8)
    dq, dk, dv = new(B, T, Hk, D), new(B, T, Hk, D), new(B, T, Hv, D)
    dg, dbeta, dS0 = new(B, T, Hv), new(B, T, Hv), new(B, Hv, D, D)
    L.check(lib.gdn_bwd(p(q), p(k), p(v), p(g), p(beta), p(state), p(mask), p(saved), saved.numel(), p(dy), None, p(dq),
                        p(dk), p(dv), p(dg), p(dbeta), p(dS0), p(wb), wb.numel(), *shape, code, L.DTYPE_CODE[dy_dtype], L.F32,
                        gate, form, st))
    return [x.double().cpu().numpy() for x in (y, dq, dk, dg, dbeta, dS0)]


def _inputs(B, T, Hk, Hv, dy_dtype, seed):
    d = O.make_inputs(B, T, Hk, Hv, D, seed=seed, s0_std=1.0)
    rnd = lambda x: torch.tensor(x).bfloat16().float().numpy()
    mask = np.zeros((B, T), bool)
    mask[:, 0] = True
    return dict(d, mask=mask, decay=np.clip(d["decay"], 0.25, None).astype(np.float32),
                **{n: rnd(d[n]) for n in "qkv"}, dy=rnd(d["dy"]) if dy_dtype == torch.bfloat16 else d["dy"])


def _oracle(d):
    (y, _), g = O.gated_delta_chunked_vjp(d["q"], d["k"], d["v"], d["decay"], d["beta"], d["state"], d["mask"], d["dy"],
                                          np.zeros_like(d["state"]), chunk=64, dtype=np.float64)
    return y, g[0], g[1], g[3], g[4], g[5]


def _off(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("dy_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,Hk,Hv,chunk", [(1, 64, 1, 4, 64), (1, 200, 2, 2, 64), (2, 70, 16, 32, 64), (4, 70, 16, 32, 64),
                                             (1, 300, 2, 4, 128), (4, 150, 16, 32, 128)])
def test_queries_that_read_an_entry_state(dev, B, T, Hk, Hv, chunk, dy_dtype):
    """beta = 0 at the unmasked token, so every output reads S0: the state's and q~'s halves in y, dq, dk, dg, dbeta and
    dS0, at slices of 16, 32 and 64 value channels, in whole and in rebuilt windows; in one chunk also q~'s in the dg of the
    unmasked token (further on that also takes the state's adjoint, a bf16 tile)."""
    d = _inputs(B, T, Hk, Hv, dy_dtype, seed=T + Hv)
    d["beta"][:, 0] = 0.0
    got, want = _call(d, dev, chunk, dy_dtype), _oracle(d)
    for name, a, b in zip(("y", "dq", "dk", "dg", "dbeta"), got, want):
        assert _off(a[:, 1:], b[:, 1:]) <= BAR, name
    assert _off(got[5], want[5]) <= BAR, "dS0"
    if T <= 64:
        assert _off(got[3][:, 0], want[3][:, 0]) <= BAR, "dg of the unmasked token"


@pytest.mark.parametrize("dy_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,Hk,Hv", [(1, 64, 1, 4), (1, 63, 2, 2), (4, 64, 16, 32)])
def test_queries_that_read_a_key(dev, B, T, Hk, Hv, dy_dtype):
    """No state before the unmasked token: the others read its key through P = q~ K^T, and its dk is dP^T q~."""
    d = _inputs(B, T, Hk, Hv, dy_dtype, seed=T)
    d["state"] = np.zeros_like(d["state"])
    got, want = _call(d, dev, 64, dy_dtype), _oracle(d)
    # the part of y that P gives: without beta c v, which is added in fp32
    rep = lambda x: np.repeat(x.astype(np.float64), Hv // Hk, axis=2)
    ev = (d["beta"] * (rep(d["q"]) * rep(d["k"])).sum(-1))[..., None].astype(np.float64) * d["v"]
    assert _off((got[0] - ev)[:, 1:], (want[0] - ev)[:, 1:]) <= BAR, "y"
    for name, a, b in zip(("dq", "dk", "dg", "dbeta"), got[1:], want[1:]):
        assert _off(a[:, 1:], b[:, 1:]) <= BAR, name
    assert _off(got[2][:, 0], want[2][:, 0]) <= BAR, "dk of the unmasked token"


def test_groups_keep_both_halves(dev):
    """Groups of 2048 chunk-heads, forward-only and checkpointed, against the call in one piece: the first group ends at
    token 512 of 600."""
    import gdn_engine
    d = _inputs(1, 600, 64, 256, torch.float32, seed=9)
    d["beta"][:, 0] = 0.0
    whole, groups = _call(d, dev, 64, torch.float32), _call(d, dev, 128, torch.float32)
    for name, a, b in zip(("y", "dq", "dk", "dg", "dbeta"), groups, whole):
        assert _off(a[:, 1:], b[:, 1:]) <= BAR, name
    assert _off(groups[5], whole[5]) <= BAR, "dS0"
    t = lambda n, dt=torch.float32: torch.tensor(d[n], device=dev).to(dt)
    y, _ = gdn_engine.recurrence(*(t(n, torch.bfloat16) for n in "qkv"), t("decay"), t("beta"), t("state"),
                                 t("mask", torch.bool), need_grad=False, output_dtype=torch.float32)
    assert _off(y.double().cpu().numpy()[:, 1:], whole[0][:, 1:]) <= BAR, "y of the forward-only call"

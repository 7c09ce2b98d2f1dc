"""Masked calls on the chunked form where their kernels branch: chunks with no, one (first / last row), some and only
masked tokens beside each other, one, two and four value heads per key head, each input dtype and both gate conventions,
against the fp64 oracle; and group-wise calls (forward-only, checkpointed) against whole ones.

Tolerances: fp32 outputs of fp32 / fp16 inputs 1e-4 as in the other parity tests; bf16 contractions 1e-2."""

import numpy as np
import pytest
import torch

from oracle import gdn_oracle as O

pytestmark = pytest.mark.gpu

D = 128
NAMES = ("y", "S_T", "dq", "dk", "dv", "dg", "dbeta", "dS0")
DT = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gdn_lib
    gdn_lib.load()
    return torch.device("cuda:0")


def _mask(B, T, rng):
    m = np.ones((B, T), bool)
    m[0, 64:128] = False                      # a whole chunk masked between two that are not
    m[0, 192:193] = False                     # a chunk's first row only
    m[-1, 63:64] = False                      # a chunk's last row only
    m[-1, T - 1:] = False                     # the sequence's last token
    m[-1, 128:192] = rng.random(64)[: max(0, min(192, T) - 128)] > 0.5 if T >= 192 else m[-1, 128:192]
    return m


def _run(d, dev, dtype, log_gate, y_dtype, chunk=64):
    import gdn_engine
    t = lambda x, dt=torch.float32: torch.tensor(x, device=dev, dtype=dt).requires_grad_(True)
    xs = [t(d[n], DT[dtype]) for n in "qkv"] + [t(d["g_log" if log_gate else "decay"]), t(d["beta"]), t(d["state"])]
    y, S = gdn_engine.recurrence(*xs, torch.tensor(d["mask"], device=dev), chunk, log_gate=log_gate, output_dtype=y_dtype)
    g = torch.autograd.grad([y, S], xs, [torch.tensor(d["dy"], device=dev, dtype=y_dtype), torch.tensor(d["dS_T"], device=dev)])
    return [x.detach().double().cpu().numpy() for x in (y, S, *g)]


@pytest.mark.parametrize("dtype,y_dtype,rep,log_gate,T", [
    ("fp32", "fp32", 2, False, 257), ("fp32", "fp32", 1, True, 200), ("fp16", "fp32", 4, False, 200),
    ("bf16", "bf16", 2, True, 257), ("bf16", "fp32", 4, False, 200), ("bf16", "bf16", 1, False, 193)])
def test_masked_chunks_of_every_kind(dev, dtype, y_dtype, rep, log_gate, T):
    B, Hk = 2, 2
    rng = np.random.default_rng(T + rep)
    d = O.make_inputs(B, T, Hk, Hk * rep, D, seed=T, s0_std=0.05)
    rnd = lambda x, dt: torch.tensor(x).to(DT[dt]).float().numpy()
    d = dict(d, mask=_mask(B, T, rng), dS_T=(0.1 * rng.standard_normal(d["state"].shape)).astype(np.float32),
             q=rnd(d["q"], dtype), k=rnd(d["k"], dtype), v=rnd(d["v"], dtype), dy=rnd(d["dy"], y_dtype))
    got = _run(d, dev, dtype, log_gate, DT[y_dtype])
    (wy, wS), wg = O.gated_delta_chunked_vjp(d["q"], d["k"], d["v"], d["decay"], d["beta"], d["state"], d["mask"], d["dy"],
                                             d["dS_T"], chunk=64, dtype=np.float64)
    if log_gate:
        wg = (*wg[:3], wg[3] * d["decay"], *wg[4:])
    for name, a, b in zip(NAMES, got, (wy, wS, *wg)):
        # dq, dk, dv come back in the inputs' dtype: fp16 rounds them by up to 2^-11
        bar = 1e-2 if dtype == "bf16" else 1e-3 if dtype == "fp16" and name in ("dq", "dk", "dv") else 1e-4
        assert np.abs(a - b).max() <= bar * np.abs(b).max(), name


@pytest.mark.parametrize("dtype,y_dtype,log_gate", [("fp32", "fp32", False), ("fp16", "fp32", True), ("bf16", "bf16", True)])
def test_masked_chunks_of_every_kind_at_wide_slices(dev, dtype, y_dtype, log_gate):
    """128 heads take 64-wide slices in the sequential kernels: training, checkpointed and forward-only calls."""
    import gdn_engine
    B, T, Hk, Hv = 4, 200, 16, 32
    rng = np.random.default_rng(T)
    d = O.make_inputs(B, T, Hk, Hv, D, seed=T, s0_std=0.05)
    rnd = lambda x, dt: torch.tensor(x).to(DT[dt]).float().numpy()
    d = dict(d, mask=_mask(B, T, rng), dS_T=(0.1 * rng.standard_normal(d["state"].shape)).astype(np.float32),
             q=rnd(d["q"], dtype), k=rnd(d["k"], dtype), v=rnd(d["v"], dtype), dy=rnd(d["dy"], y_dtype))
    (wy, wS), wg = O.gated_delta_chunked_vjp(d["q"], d["k"], d["v"], d["decay"], d["beta"], d["state"], d["mask"], d["dy"],
                                             d["dS_T"], chunk=64, dtype=np.float64)
    if log_gate:
        wg = (*wg[:3], wg[3] * d["decay"], *wg[4:])
    want = (wy, wS, *wg)
    with torch.no_grad():
        t = lambda x, dt=torch.float32: torch.tensor(x, device=dev, dtype=dt)
        fwd = gdn_engine.recurrence(*(t(d[n], DT[dtype]) for n in "qkv"), t(d["g_log" if log_gate else "decay"]), t(d["beta"]),
                                    t(d["state"]), t(d["mask"], torch.bool), log_gate=log_gate, output_dtype=DT[y_dtype],
                                    need_grad=False)
    for got in (_run(d, dev, dtype, log_gate, DT[y_dtype]), _run(d, dev, dtype, log_gate, DT[y_dtype], chunk=128),
                [x.double().cpu().numpy() for x in fwd]):
        for name, a, b in zip(NAMES, got, want):
            bar = 1e-2 if dtype == "bf16" else 1e-3 if dtype == "fp16" and name in ("dq", "dk", "dv") else 1e-4
            assert np.abs(a - b).max() <= bar * np.abs(b).max(), name


@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
def test_masked_groups_equal_whole_calls(dev, dtype):
    """Groups of 2048 chunk-heads: 64 heads x 2200 tokens take two groups, forward-only and checkpointed."""
    import gdn_engine
    B, T, Hk, Hv = 2, 2200, 16, 32
    gen = torch.Generator(device=dev).manual_seed(3)
    n = lambda *s: torch.randn(*s, device=dev, generator=gen)
    unit = lambda x: x * torch.rsqrt((x * x).sum(-1, keepdim=True))
    xs = [(unit(n(B, T, Hk, D)) * D ** -0.5).to(DT[dtype]), unit(n(B, T, Hk, D)).to(DT[dtype]), n(B, T, Hv, D).to(DT[dtype]),
          -torch.rand(B, T, Hv, device=dev, generator=gen), torch.rand(B, T, Hv, device=dev, generator=gen),
          0.1 * n(B, Hv, D, D)]
    mask = torch.arange(T, device=dev)[None] < torch.tensor([[2070], [700]], device=dev)
    mask[1, 5] = False
    xs = [x.requires_grad_(True) for x in xs]
    dy, dS = n(B, T, Hv, D), n(B, Hv, D, D)
    outs = {}
    for chunk in (64, 256):
        y, S = gdn_engine.recurrence(*xs, mask, chunk, log_gate=True, output_dtype=torch.float32)
        outs[chunk] = [y, S, *torch.autograd.grad([y, S], xs, [dy, dS])]
    y, S = gdn_engine.recurrence(*xs, mask, 64, log_gate=True, output_dtype=torch.float32, need_grad=False)
    # the same arithmetic per chunk; the states that enter a group are carried in fp32 in each form
    bar = 1e-2 if dtype == "bf16" else 1e-5
    for name, a, b in [*zip(NAMES, outs[256], outs[64]), ("y", y, outs[64][0]), ("S_T", S, outs[64][1])]:
        assert float((a - b).detach().abs().max()) <= bar * float(b.detach().abs().max()), name

"""Performance cases: the calls that a user's training, prefill and decode programs make, with their inputs, the work
they cannot do without, the tolerance of their results, and the results themselves in 64-bit arithmetic.

A case's ``kind`` names the entry point:

  train         forward + VJP of one layer's delta rule: ``gated_delta_chunked`` (or, with ``chunk`` > 64,
                ``gated_delta_ops_checkpointed``) on decays; with ``log_gate``, ``gdn_engine.recurrence`` on log decays
                with outputs in the inputs' type.  Returns y, the final state and every gradient.
  prefill       ``gated_delta_update(..., use_kernel=True)``: gates and forward-only recurrence, as inference and
                frozen layers run it.
  decode        ``gdn_engine.decode_step``: one token of B sequences, the states updated in place.
  block         forward + backward of a whole GDN block with LoRA adapters on its projections.
  block_decode  one token of B sequences through a whole block with its conv and recurrent caches.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch
import torch.nn.functional as F

_PKG = str(Path(__file__).resolve().parent.parent / "moe-stream-mac_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import gated_delta  # noqa: E402
import gdn_checkpoint  # noqa: E402
import gdn_engine  # noqa: E402
import gdn_vjp  # noqa: E402
import qwen3_5  # noqa: E402

DEV = "cuda"
TORCH_DTYPE = {"bf16": torch.bfloat16, "fp32": torch.float32}
HEADS = dict(Hk=16, Hv=32, D=128)  # the layer the benchmark measures
LORA_RANK, LORA_SCALE = 16, 20.0


def _train(name, **kw):
    c = dict(name=name, kind="train", B=1, T=64, **HEADS, dtype="bf16", chunk=64, gate="head", log_gate=False,
             mask=False, s0=False)
    c.update(kw)
    return c


def listed():
    return [
        # one generated token of one sequence through a block: what an interactive user waits for
        dict(name="block_decode_b1", kind="block_decode", B=1, hidden=2048, **HEADS),
        # one decode step of a serving batch
        dict(name="decode_bf16_b64", kind="decode", B=64, **HEADS, dtype="bf16"),
        # a short fp32 sequence: launches and host time count
        _train("train_fp32_b1_t64", dtype="fp32", T=64),
        # a small model with 64-wide heads (the sizes a first experiment uses)
        _train("train_fp32_b4_t512_d64", dtype="fp32", B=4, T=512, Hk=4, Hv=8, D=64),
        # fp32 training from a carried state, with its gradient
        _train("train_fp32_b1_t2048_s0", dtype="fp32", T=2048, s0=True),
        # one bf16 sequence of odd length through the drop-in call
        _train("train_bf16_b1_t4001", T=4001),
        # the benchmark's batch: bf16 in and out, log decays
        _train("train_bf16_b4_t4096", B=4, T=4096, log_gate=True),
        # a padded batch: sequences of different lengths, the padding masked
        _train("masked_bf16_b4_t4096", B=4, T=4096, mask=True),
        # one decay per key channel
        _train("channel_bf16_b4_t2048", B=4, T=2048, gate="channel"),
        # a long sequence, states kept every 256 tokens and recomputed in the backward
        _train("checkpoint_fp32_b1_t16384", dtype="fp32", T=16384, chunk=256),
        # a long prompt (or a frozen layer): forward only
        dict(name="prefill_bf16_b2_t8100", kind="prefill", B=2, T=8100, **HEADS, dtype="bf16"),
        # LoRA fine-tuning of a whole block
        dict(name="block_bf16_b2_t8192", kind="block", B=2, T=8192, hidden=2048, **HEADS),
    ]


def _logint(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["train"] * 8 + ["prefill"] * 2 + ["decode", "block", "block_decode"])
    Hk, Hv = rng.choice([(16, 32), (16, 32), (16, 16), (8, 16), (4, 16)])
    if kind == "decode":
        return dict(kind=kind, B=_logint(rng, 1, 64), Hk=Hk, Hv=Hv, D=128, dtype=rng.choice(["bf16", "bf16", "fp32"]))
    if kind == "block_decode":
        return dict(kind=kind, B=_logint(rng, 1, 32), hidden=rng.choice([1024, 2048]), Hk=Hk, Hv=Hv, D=128)
    if kind == "block":
        B = rng.choice([1, 2, 4])
        return dict(kind=kind, B=B, T=_logint(rng, 256, 16384 // B), hidden=rng.choice([1024, 2048]), Hk=Hk, Hv=Hv,
                    D=128)
    B = rng.choice([1, 1, 2, 3, 4, 8])
    dtype = rng.choice(["bf16", "bf16", "fp32"])
    if kind == "prefill":
        return dict(kind=kind, B=B, T=_logint(rng, 16, 16384 // B), Hk=Hk, Hv=Hv, D=128, dtype=dtype)
    D = rng.choice([128] * 6 + [64, 32])
    gate = rng.choice(["head"] * 4 + ["channel"])
    mask = rng.random() < 0.25
    cap = 16384 * 32  # head-tokens
    if dtype == "fp32":
        cap //= 2
    if D < 128 or (gate == "channel" and (dtype == "fp32" or mask)):
        cap //= 4
    T = _logint(rng, 16, max(16, min(8192, cap // (B * Hv))))
    return dict(kind=kind, B=B, T=T, Hk=Hk, Hv=Hv, D=D, dtype=dtype, chunk=rng.choice([64, 64, 64, 256]), gate=gate,
                log_gate=dtype == "bf16" and rng.random() < 0.3, mask=mask, s0=rng.random() < 0.4)


# ------------------------------------------------------------------------------------------------ inputs


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _inputs(case, seed):
    """q, k, v, gate inputs, beta, state and cotangent with the layer's distributions (k and q unit rows, q scaled)."""
    gen = _gen(seed)
    n = lambda *s: torch.randn(*s, device=DEV, generator=gen)
    B, T, Hk, Hv, D = case["B"], case.get("T", 1), case["Hk"], case["Hv"], case["D"]
    dt = TORCH_DTYPE[case.get("dtype", "bf16")]
    unit = lambda x: x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)
    A_log = torch.empty(Hv, device=DEV).uniform_(0.0, math.log(16.0), generator=gen)
    channel = case.get("gate") == "channel"
    a = n(B, T, Hv, D) if channel else n(B, T, Hv)
    glog = -torch.exp(A_log)[:, None] * F.softplus(a) if channel else -torch.exp(A_log) * F.softplus(a)
    mask = None
    if case.get("mask"):  # right padding: lengths from half of T to T, the longest sequence whole
        lens = torch.randint((T + 1) // 2, T + 1, (B,), device=DEV, generator=gen)
        lens[0] = T
        mask = torch.arange(T, device=DEV)[None, :] < lens[:, None]
        if B == 1:
            mask[:, T - T // 8:] = False
    s0 = case.get("s0") or case["kind"] in ("decode", "block_decode")
    return dict(q=(unit(n(B, T, Hk, D)) * D ** -0.5).to(dt), k=unit(n(B, T, Hk, D)).to(dt), v=n(B, T, Hv, D).to(dt),
                glog=glog, a=a, b=n(B, T, Hv), A_log=A_log, dt_bias=torch.zeros(Hv, device=DEV), mask=mask,
                state=n(B, Hv, D, D) * 0.02 if s0 else None, dy=n(B, T, Hv, D))


def _block_inputs(case, seed):
    """The block, its input and (training) the output's cotangent, or (decode) the caches after a prompt."""
    torch.manual_seed(seed)
    gen = _gen(seed + 1)
    args = qwen3_5.ModelArgs(hidden_size=case["hidden"], linear_num_key_heads=case["Hk"],
                             linear_num_value_heads=case["Hv"], linear_key_head_dim=case["D"],
                             linear_value_head_dim=case["D"])
    n = lambda *s: torch.randn(*s, device=DEV, generator=gen)
    with torch.device("meta"):
        blk = qwen3_5.GatedDeltaNet(args)
    blk = blk.to_empty(device=DEV)
    projs = ("in_proj_qkv", "in_proj_z", "in_proj_b", "in_proj_a", "out_proj")
    with torch.no_grad():
        for m in projs:
            getattr(blk, m).weight.copy_(0.02 * n(*getattr(blk, m).weight.shape))
        blk.conv1d.weight.copy_(0.25 * n(*blk.conv1d.weight.shape))
        blk.A_log.uniform_(0.0, math.log(16.0), generator=gen)
        blk.dt_bias.zero_()
        blk.norm.weight.copy_(1 + 0.1 * n(*blk.norm.weight.shape))
    qwen3_5.freeze(blk)
    B = case["B"]
    if case["kind"] == "block_decode":
        blk = blk.to(torch.bfloat16).eval()
        return blk, dict(x=n(B, 1, case["hidden"]).to(torch.bfloat16), conv=n(B, blk.K - 1, blk.conv_dim),
                         state=0.02 * n(B, case["Hv"], case["D"], case["D"]))
    for m in projs:
        lin = qwen3_5.LoRALinear(getattr(blk, m), LORA_RANK, LORA_SCALE)
        lin.lora_a = torch.nn.Parameter(0.02 * n(*lin.lora_a.shape))
        lin.lora_b = torch.nn.Parameter(0.002 * n(*lin.lora_b.shape))  # some steps into the training
        setattr(blk, m, lin)
    blk = blk.to(torch.bfloat16).train()
    shape = (B, case["T"], case["hidden"])
    return blk, dict(x=n(*shape).to(torch.bfloat16), dout=n(*shape).to(torch.bfloat16))


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("block", "block_decode"):
        blk, x = _block_inputs(case, seed)
        if kind == "block":
            # gdn_vjp.install()'s update is what the block's training call resolves to
            gdn_vjp.install()
            x["x"].requires_grad_(True)
            x["names"] = ["x"] + [k for k, p in blk.named_parameters() if p.requires_grad]
            x["leaves"] = [x["x"]] + [p for p in blk.parameters() if p.requires_grad]
        return dict(case=case, blk=blk, **x)
    x = _inputs(case, seed)
    if kind == "decode":
        x = {k: (t[:, 0].contiguous() if k in ("q", "k", "v", "glog", "b") else t) for k, t in x.items()}
        return dict(case=case, q=x["q"], k=x["k"], v=x["v"], g=x["glog"], beta=torch.sigmoid(x["b"]),
                    state=x["state"])
    if kind == "prefill":
        dt = TORCH_DTYPE[case["dtype"]]
        return dict(case=case, q=x["q"], k=x["k"], v=x["v"], a=x["a"].to(dt), b=x["b"].to(dt), A_log=x["A_log"],
                    dt_bias=x["dt_bias"])
    log_gate = case["log_gate"]
    leaves = dict(q=x["q"], k=x["k"], v=x["v"], g=x["glog"] if log_gate else torch.exp(x["glog"]),
                  beta=torch.sigmoid(x["b"]))
    state = x["state"]
    if log_gate and state is None:
        B, Hv, D = case["B"], case["Hv"], case["D"]
        state = torch.zeros(B, Hv, D, D, device=DEV)
    if case["s0"]:
        leaves["state"] = state
    for t in leaves.values():
        t.requires_grad_(True)
    dy = x["dy"].to(TORCH_DTYPE[case["dtype"]]) if log_gate else x["dy"]
    return dict(case=case, leaves=leaves, state=state, mask=x["mask"], dy=dy)


# ------------------------------------------------------------------------------------------------ one pass


def run(s):
    kind = s["case"]["kind"]
    if kind == "decode":
        y = gdn_engine.decode_step(s["q"], s["k"], s["v"], s["g"], s["beta"], s["state"], s["state"], log_gate=True,
                                   out_dtype=s["q"].dtype)
        return dict(y=y, state=s["state"])
    if kind == "prefill":
        with torch.no_grad():
            y, S = gated_delta.gated_delta_update(s["q"], s["k"], s["v"], s["a"], s["b"], s["A_log"], s["dt_bias"],
                                                  use_kernel=True)
        return dict(y=y, state=S)
    if kind == "block_decode":
        cache = qwen3_5.GDNCache()
        cache[0], cache[1] = s["conv"], s["state"]
        with torch.no_grad():
            out = s["blk"](s["x"], cache=cache)
        return dict(out=out, conv=cache[0], state=cache[1])
    if kind == "block":
        out = s["blk"](s["x"])
        grads = torch.autograd.grad(out, s["leaves"], s["dout"])
        return dict(out=out, **{"d_" + n: g for n, g in zip(s["names"], grads)})
    c, x = s["case"], s["leaves"]
    args = (x["q"], x["k"], x["v"], x["g"], x["beta"], s["state"], s["mask"])
    if c["log_gate"]:
        y, S = gdn_engine.recurrence(*args, chunk=c["chunk"], log_gate=True, output_dtype=x["q"].dtype)
    elif c["chunk"] > 64:
        y, S = gdn_checkpoint.gated_delta_ops_checkpointed(*args, chunk=c["chunk"])
    else:
        y, S = gdn_vjp.gated_delta_chunked(*args, chunk=c["chunk"])
    grads = torch.autograd.grad([y], list(x.values()), [s["dy"]])
    return dict(y=y, S=S, **{"d" + n: g for n, g in zip(x, grads)})


# ------------------------------------------------------------------------------------------------ work, tolerance


def work(case):
    B, T, Hk, Hv, D = case["B"], case.get("T", 1), case["Hk"], case["Hv"], case["D"]
    kind, tok = case["kind"], case["B"] * case.get("T", 1)
    e = 2 if case.get("dtype", "bf16") == "bf16" else 4
    states = 4 * B * Hv * D * D
    if kind == "decode":
        return dict(bytes=2 * states + tok * (e * 2 * (Hk + Hv) * D + 8 * Hv), flops=7 * tok * Hv * D * D)
    if kind == "prefill":
        return dict(bytes=states + tok * (e * (2 * Hk + Hv) * D + 4 * Hv * D + 2 * e * Hv), flops=7 * tok * Hv * D * D)
    if kind in ("block", "block_decode"):
        h, conv = case["hidden"], (2 * Hk + Hv) * D
        weights = h * (conv + 2 * Hv * D + 2 * Hv)
        if kind == "block_decode":
            return dict(bytes=2 * weights + 2 * states + 8 * B * 3 * conv + 4 * B * h,
                        flops=B * (2 * weights + 7 * Hv * D * D))
        lora = LORA_RANK * (5 * h + conv + 2 * Hv * D + 2 * Hv)
        return dict(bytes=2 * (weights + 2 * lora + 4 * tok * h), flops=tok * (4 * weights + 6 * lora + 27 * Hv * D * D))
    gate = Hv * D if case["gate"] == "channel" else Hv
    out = e if case["log_gate"] else 4
    s0 = 2 * states if case["s0"] else 0
    return dict(bytes=tok * (e * (4 * Hk + 2 * Hv) * D + 2 * out * Hv * D + 8 * gate + 8 * Hv) + states + s0,
                flops=27 * tok * Hv * D * D)


def tolerance(case):
    # Against 64 bits the results are off by up to 2.4e-3 (bf16 inputs: roundings of 2^-9, a few in a row), 8.5e-3 (a
    # block, where they travel through every step) and 4.5e-7 (fp32: sums of some hundred terms, decays from exp).
    if case["kind"] in ("block", "block_decode"):
        return {"rel": 0.02, "max": 0.5}
    if case.get("dtype", "bf16") == "fp32":
        return {"rel": 3e-6, "max": 2e-4}
    return {"rel": 0.01, "max": 0.3}


# ------------------------------------------------------------------------------------------------ 64-bit results


class _Recurrence64(torch.autograd.Function):
    """The delta rule token by token in float64: y_t = S~_t q_t with S~_t = S_{t-1} d_t + delta_t k_t^T; a masked
    token keeps S_{t-1}.  States are kept every 64 tokens and recomputed in the backward.  q, k per value head."""

    SEG = 64

    @staticmethod
    def step(S, q, k, v, d, beta, keep):
        A = S * d
        r = v - torch.matmul(A, k[..., None])[..., 0]
        delta = beta * r
        cand = A + delta[..., None] * k[..., None, :]
        return A, r, delta, cand, cand if keep is None else torch.where(keep, cand, S)

    @staticmethod
    def forward(ctx, q, k, v, d, beta, S, mask):
        ctx.set_materialize_grads(False)
        step, kept, ys = _Recurrence64.step, [], []
        for t in range(q.shape[1]):
            if t % _Recurrence64.SEG == 0:
                kept.append(S)
            keep = None if mask is None else mask[:, t, None, None, None]
            _, _, _, cand, S = step(S, q[:, t], k[:, t], v[:, t], d[:, t], beta[:, t, :, None], keep)
            ys.append(torch.matmul(cand, q[:, t, ..., None])[..., 0])
        ctx.save_for_backward(q, k, v, d, beta)
        ctx.kept, ctx.mask = kept, mask
        return torch.stack(ys, 1), S

    @staticmethod
    def backward(ctx, dy, dS):
        q, k, v, d, beta = ctx.saved_tensors
        mask, seg, T = ctx.mask, _Recurrence64.SEG, q.shape[1]
        dS = torch.zeros_like(ctx.kept[0]) if dS is None else dS
        grads = [torch.empty_like(x) for x in (q, k, v, d, beta)]
        dq, dk, dv, dd, db = grads
        channel = d.shape[-1] > 1
        for first in range((T - 1) // seg * seg, -1, -seg):
            S, rows = ctx.kept[first // seg], []
            for t in range(first, min(first + seg, T)):
                keep = None if mask is None else mask[:, t, None, None, None]
                rows.append((S, keep))
                S = _Recurrence64.step(S, q[:, t], k[:, t], v[:, t], d[:, t], beta[:, t, :, None], keep)[4]
            for t in range(min(first + seg, T) - 1, first - 1, -1):
                S, keep = rows[t - first]
                qt, kt, bt = q[:, t], k[:, t], beta[:, t, :, None]
                A, r, delta, cand, _ = _Recurrence64.step(S, qt, kt, v[:, t], d[:, t], bt, keep)
                dcand = dS if keep is None else torch.where(keep, dS, 0.0)
                back = 0.0 if keep is None else torch.where(keep, 0.0, dS)
                dcand = dcand + dy[:, t, ..., None] * qt[..., None, :]
                dq[:, t] = torch.matmul(dy[:, t, ..., None, :], cand)[..., 0, :]
                ddelta = torch.matmul(dcand, kt[..., None])[..., 0]
                dvt = bt * ddelta
                dv[:, t] = dvt
                db[:, t] = (ddelta * r).sum(-1)
                dk[:, t] = (torch.matmul(delta[..., None, :], dcand) - torch.matmul(dvt[..., None, :], A))[..., 0, :]
                dA = dcand - dvt[..., None] * kt[..., None, :]
                dd[:, t] = (dA * S).sum(-2 if channel else (-2, -1), keepdim=True)
                dS = dA * d[:, t] + back
            rows = None
        return dq, dk, dv, dd, db, dS, None


def _recurrence64(q, k, v, d, beta, state, mask=None):
    """d [B, T, Hv] or [B, T, Hv, Dk] decays; q, k per key head."""
    rep = v.shape[2] // q.shape[2]
    q, k = (x.repeat_interleave(rep, 2) for x in (q, k))
    d = d[..., None, None] if d.dim() == 3 else d[..., None, :]
    if state is None:
        state = q.new_zeros(q.shape[0], v.shape[2], v.shape[3], q.shape[3])
    return _Recurrence64.apply(q, k, v, d, beta, state, mask)


def _decay64(a, A_log, dt_bias):
    return torch.exp(-torch.exp(A_log) * F.softplus(a + dt_bias, threshold=60.0))


def _block64(blk, x, conv_state, state, adapters):
    """One GDN block over x [B, T, hidden] in float64; ``adapters``: float64 (A, B) per projection, or None."""
    B, T, _ = x.shape
    Hk, Hv, D, K = blk.Hk, blk.Hv, blk.Dk, blk.K

    def proj(name, x):
        y = x @ getattr(blk, name).weight.double().t()
        if adapters:
            A, Bm = adapters[name]
            y = y + LORA_SCALE * ((x @ A.t()) @ Bm.t())
        return y

    qkv = proj("in_proj_qkv", x)
    past = qkv.new_zeros(B, K - 1, qkv.shape[-1]) if conv_state is None else conv_state.double()
    seq = torch.cat([past, qkv], 1)
    w = blk.conv1d.weight.double()[:, 0]
    c = F.silu(sum(seq[:, i:i + T] * w[:, i] for i in range(K)))
    q, k, v = c.split([Hk * D, Hk * D, Hv * D], -1)
    unit = lambda t, s: t * (s * torch.rsqrt((t * t).sum(-1, keepdim=True) + 1e-6))
    q, k = unit(q.reshape(B, T, Hk, D), D ** -0.5), unit(k.reshape(B, T, Hk, D), 1.0)
    d = _decay64(proj("in_proj_a", x), blk.A_log.double(), blk.dt_bias.double())
    y, S = _recurrence64(q, k, v.reshape(B, T, Hv, D), d, torch.sigmoid(proj("in_proj_b", x)), state)
    z = proj("in_proj_z", x).reshape(B, T, Hv, D)
    o = y * torch.rsqrt((y * y).mean(-1, keepdim=True) + blk.norm.eps) * blk.norm.weight.double() * F.silu(z)
    return proj("out_proj", o.reshape(B, T, Hv * D)), seq[:, T:], S


def exact(case, seed):
    kind = case["kind"]
    if kind == "block_decode":
        blk, x = _block_inputs(case, seed)
        with torch.no_grad():
            out, conv, S = _block64(blk, x["x"].double(), x["conv"], x["state"].double(), None)
        return dict(out=out, conv=conv, state=S)
    if kind == "block":
        blk, x = _block_inputs(case, seed)
        xd = x["x"].double().requires_grad_(True)
        names, leaves, adapters = ["x"], [xd], {}
        for n, p in blk.named_parameters():
            if p.requires_grad:
                names.append(n)
                leaves.append(p.detach().double().requires_grad_(True))
                m, which = n.rsplit(".", 1)
                adapters.setdefault(m, [None, None])[which == "lora_b"] = leaves[-1]
        out, _, _ = _block64(blk, xd, None, None, adapters)
        grads = torch.autograd.grad(out, leaves, x["dout"].double())
        return dict(out=out.detach(), **{"d_" + n: g for n, g in zip(names, grads)})
    x = {k: (t.double() if torch.is_tensor(t) and t.dtype != torch.bool else t)
         for k, t in _inputs(case, seed).items()}
    if kind == "prefill":
        dt = TORCH_DTYPE[case["dtype"]]
        d = _decay64(x["a"].to(dt).double(), x["A_log"], x["dt_bias"])
        with torch.no_grad():
            y, S = _recurrence64(x["q"], x["k"], x["v"], d, torch.sigmoid(x["b"].to(dt).double()), None)
        return dict(y=y, state=S)
    if kind == "decode":
        beta = torch.sigmoid(x["b"].float()).double()
        with torch.no_grad():
            y, S = _recurrence64(x["q"], x["k"], x["v"], torch.exp(x["glog"]), beta, x["state"])
        return dict(y=y[:, 0], state=S)
    log_gate = case["log_gate"]
    g = x["glog"] if log_gate else torch.exp(x["glog"].float()).double()
    leaves = dict(q=x["q"], k=x["k"], v=x["v"], g=g, beta=torch.sigmoid(x["b"].float()).double())
    if case["s0"]:
        leaves["state"] = x["state"]
    for t in leaves.values():
        t.requires_grad_(True)
    y, S = _recurrence64(leaves["q"], leaves["k"], leaves["v"], torch.exp(g) if log_gate else g, leaves["beta"],
                         x["state"], x["mask"])
    dy = x["dy"].to(TORCH_DTYPE[case["dtype"]]).double() if log_gate else x["dy"]
    grads = torch.autograd.grad([y], list(leaves.values()), [dy])
    return dict(y=y.detach(), S=S.detach(), **{"d" + n: t for n, t in zip(leaves, grads)})

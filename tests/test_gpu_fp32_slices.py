"""The fp32 sequential kernels at each value-slice width (16, 32 and 64 wide, chosen by the number of heads), at the edges
of a chunk, with fp32 and with fp16 inputs (the two instantiations of each), whole and with recomputed windows, against the
fp64 oracle.

Tolerances: fp32 results 1e-4 of the largest value as in the other parity tests; fp16 results round by up to 2^-11."""

import numpy as np
import pytest
import torch

from oracle import gdn_oracle as O

pytestmark = pytest.mark.gpu

D = 128
NAMES = ("y", "S_T", "dq", "dk", "dv", "dg", "dbeta", "dS0")


@pytest.mark.parametrize("dtype", ["fp32", "fp16"])
@pytest.mark.parametrize("B,Hk,Hv,T,chunk", [
    (1, 1, 2, 1, 64), (1, 2, 2, 63, 64), (1, 1, 2, 64, 64), (1, 2, 4, 65, 64), (3, 1, 3, 193, 64),     # 16 wide
    (2, 16, 32, 66, 64), (4, 16, 16, 127, 64),                                                         # 32 wide
    (4, 16, 32, 65, 64), (8, 16, 16, 129, 64),                                                         # 64 wide
    (1, 2, 4, 385, 128), (2, 16, 32, 200, 128), (4, 16, 32, 140, 128),   # windows recomputed side by side
    (1, 1, 4, 100, 64), (4, 16, 32, 200, 64), (3, 16, 32, 400, 64),      # 4, 256 and 336 (chunk, key head) pairs
])
def test_slice_widths(B, Hk, Hv, T, chunk, dtype):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gdn_engine
    dev = torch.device("cuda:0")
    dt = {"fp32": torch.float32, "fp16": torch.float16}[dtype]
    d = O.make_inputs(B, T, Hk, Hv, D, seed=T + Hv, s0_std=0.05)
    rng = np.random.default_rng(T)
    for n in "qkv":
        d[n] = torch.tensor(d[n]).to(dt).float().numpy()
    dS = (0.1 * rng.standard_normal(d["state"].shape)).astype(np.float32)
    t = lambda n, dt=torch.float32: torch.tensor(d[n], device=dev, dtype=dt).requires_grad_(True)
    xs = [*(t(n, dt) for n in "qkv"), t("decay"), t("beta"), t("state")]
    y, S = gdn_engine.recurrence(*xs, None, chunk, output_dtype=torch.float32)
    g = torch.autograd.grad([y, S], xs, [torch.tensor(d["dy"], device=dev), torch.tensor(dS, device=dev)])
    got = [x.detach().double().cpu().numpy() for x in (y, S, *g)]
    (wy, wS), wg = O.gated_delta_chunked_vjp(d["q"], d["k"], d["v"], d["decay"], d["beta"], d["state"], None, d["dy"], dS,
                                             chunk=64, dtype=np.float64)
    for name, a, b in zip(NAMES, got, (wy, wS, *wg)):
        bar = 1e-3 if dtype == "fp16" and name in ("dq", "dk", "dv") else 1e-4
        assert np.abs(a - b).max() <= bar * np.abs(b).max(), name

"""The decomposition the chunked form uses for masked steps, on the CPU in float64 against the oracle's masked recurrence
(tools/gdn_vjp.py:3-6, _step_parts :238-256): one unmasked pass over the effective gates (decay 1 and beta 0 where the
mask is 0) with the query d (q - beta c k), c = k . q, at the masked tokens, beta c v added to y there, and the masked
tokens' gradients from X, the gradient of that query (gdn_mask.hip states the formulas)."""

import numpy as np
import pytest

from oracle import gdn_oracle as O


def _one_pass(d, mask, dy, dS_T, chunk, log_gate):
    q, k, v, g, beta = (d[n] for n in ("q", "k", "v", "decay", "beta"))
    rep = v.shape[2] // q.shape[2]
    m = mask[:, :, None]
    qe, ke = (np.repeat(x, rep, axis=2) for x in (q, k))
    c = (qe * ke).sum(-1)
    e = beta * c
    qt = np.where(m[..., None], qe, g[..., None] * (qe - e[..., None] * ke))
    g2, b2 = np.where(m, g, 1.0), np.where(m, beta, 0.0)
    (y, S), (X, dk, dv, dg, db, dS0) = O.gated_delta_chunked_vjp(qt, ke, v, g2, b2, d["state"], None, dy, dS_T, chunk,
                                                                 np.float64)
    y = y + np.where(m[..., None], 0.0, e[..., None] * v)
    kx, qx = (ke * X).sum(-1), (qe * X).sum(-1)
    u = (v * dy).sum(-1) - g * kx
    dq_m = g[..., None] * X + (beta * u)[..., None] * ke
    dk_m = (beta * u)[..., None] * qe - (g * e)[..., None] * X
    mm = m[..., None]
    fold = lambda x: x.reshape(*q.shape[:3], rep, -1).sum(3)
    dg = np.where(m, dg, qx - e * kx)
    return y, S, (fold(np.where(mm, X, dq_m)), fold(np.where(mm, dk, dk_m)), np.where(mm, dv, e[..., None] * dy),
                  dg * g if log_gate else dg, np.where(m, db, c * u), dS0)


@pytest.mark.parametrize("rep,chunk,log_gate", [(1, 4, False), (2, 64, True), (4, 8, False)])
def test_query_rows_match_masked_oracle(rep, chunk, log_gate):
    B, T, Hk, D = 3, 23, 2, 8
    d = O.make_inputs(B, T, Hk, Hk * rep, D, seed=5 + chunk, s0_std=0.3, dtype=np.float64)
    rng = np.random.default_rng(rep)
    mask = rng.uniform(size=(B, T)) > 0.35
    mask[0, :3] = False
    mask[1, -5:] = False
    mask[2] = False
    dS_T = rng.standard_normal(d["state"].shape)
    (wy, wS), wg = O.gated_delta_chunked_vjp(d["q"], d["k"], d["v"], d["decay"], d["beta"], d["state"], mask, d["dy"],
                                             dS_T, chunk, np.float64)
    if log_gate:
        wg = (*wg[:3], wg[3] * d["decay"], *wg[4:])
    y, S, g = _one_pass(d, mask, d["dy"], dS_T, chunk, log_gate)
    for name, a, b in [("y", y, wy), ("S_T", S, wS)] + list(zip(("dq", "dk", "dv", "dg", "dbeta", "dS0"), g, wg)):
        assert np.abs(a - b).max() <= 1e-11 * max(np.abs(b).max(), 1e-30), name

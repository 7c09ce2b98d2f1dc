"""Whether a block's update ends in the package's own (which lets one token take the fused decode), after install()
calls in any order.  CPU only."""

import importlib

import pytest


@pytest.mark.timeout(60)
@pytest.mark.parametrize("order,own", [
    ((), True), (("gdn_vjp",), True), (("gdn_checkpoint", "gdn_vjp"), True), (("gdn_vjp", "gdn_vjp"), True),
    # the third install binds over a chain that already holds its module: the two call each other
    (("gdn_vjp", "gdn_checkpoint", "gdn_vjp"), False),
    (("gdn_checkpoint", "gdn_vjp", "gdn_checkpoint", "gdn_vjp"), False)])
def test_installs_over_each_other(monkeypatch, order, own):
    import gated_delta
    import gdn_hf
    import qwen3_5
    mods = {n: importlib.import_module(n) for n in ("gdn_vjp", "gdn_checkpoint")}
    monkeypatch.setattr(qwen3_5, "gated_delta_update", gated_delta.gated_delta_update)
    monkeypatch.setattr(gdn_hf, "_hf_modules", lambda: [])
    monkeypatch.setattr(gdn_hf, "_ROUTE", dict(gdn_hf._ROUTE))
    for m in mods.values():
        monkeypatch.setattr(m, "_ORIGINAL_UPDATE", None)
    for n in order:
        mods[n].install()
    assert qwen3_5._own_update(qwen3_5.gated_delta_update) is own


def test_another_update_is_not_own(monkeypatch):
    import gdn_vjp
    import qwen3_5
    assert not qwen3_5._own_update(lambda *a, **k: None)
    monkeypatch.setattr(gdn_vjp, "_ORIGINAL_UPDATE", None)
    assert not qwen3_5._own_update(gdn_vjp._vjp_update)

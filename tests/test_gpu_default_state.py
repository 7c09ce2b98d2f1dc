"""Calls without an entry state (no state tensor reaches the kernels, no exit gradient is formed for it) give the same bits
as calls from a state of zeros, through each drop-in entry point and form: trained, forward-only, checkpointed and masked
calls, one token and none."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(B, T, Hk, Hv, D, dtype, channel, dev):
    gen = torch.Generator(device=dev).manual_seed(T)
    n = lambda *s: torch.randn(*s, device=dev, generator=gen)
    unit = lambda x: x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)
    g = torch.rand(B, T, Hv, *([D] if channel else []), device=dev, generator=gen)
    return [unit(n(B, T, Hk, D)).to(dtype), unit(n(B, T, Hk, D)).to(dtype), n(B, T, Hv, D).to(dtype), 0.5 + 0.5 * g,
            torch.rand(B, T, Hv, device=dev, generator=gen)]


@pytest.mark.parametrize("T", [0, 1, 65, 300])
@pytest.mark.parametrize("D,dtype,channel", [(128, torch.float32, False), (128, torch.bfloat16, False),
                                             (128, torch.bfloat16, True), (32, torch.float32, False)])
def test_no_state_is_a_state_of_zeros(T, D, dtype, channel):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gated_delta
    import gdn_checkpoint
    import gdn_vjp
    dev = torch.device("cuda:0")
    B, Hk, Hv = 2, 1, 2
    xs = [x.requires_grad_(True) for x in _inputs(B, T, Hk, Hv, D, dtype, channel, dev)]
    zeros = torch.zeros(B, Hv, D, D, device=dev)
    mask = torch.arange(T, device=dev)[None].expand(B, T) % 3 != 1
    calls = [lambda s: gdn_vjp.gated_delta_chunked(*xs, s), lambda s: gdn_vjp.gated_delta_chunked(*xs, s, mask),
             lambda s: gdn_checkpoint.gated_delta_ops_checkpointed(*xs, s, chunk=128), lambda s: gated_delta.gated_delta_ops(*xs, s)]
    for call in calls:
        outs = []
        for s in (None, zeros, zeros.clone().requires_grad_(True)):
            y, S = call(s)
            assert y.dtype == torch.float32 and S.dtype == torch.float32
            outs.append([y, S, *torch.autograd.grad([y, S], xs, [torch.ones_like(y), torch.ones_like(S)])])
        for other in outs[1:]:
            assert all(torch.equal(a, b) for a, b in zip(outs[0], other))
    a, b = gated_delta.gated_delta_kernel(*xs), gated_delta.gated_delta_kernel(*xs, zeros)
    assert all(torch.equal(x, y) for x, y in zip(a, b))

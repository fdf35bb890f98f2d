"""Backward passes through one of the two outputs: an output without a cotangent counts as one whose cotangent is zero,
bit for bit, with and without an initial state, in the trainable recurrence and in the fused prologue."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("carried", [True, False], ids=["state", "no_state"])
@pytest.mark.parametrize("kind", ["float32", "bf16", "prologue"])
def test_one_output(kind, carried):
    import torch
    import torch.nn.functional as F

    from quotebound_amd import gdn

    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    B, T, Hk, Hv, D = 2, 70, 2, 4, 128
    gen = torch.Generator(device="cuda").manual_seed(50)
    r = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    dt = torch.float32 if kind == "float32" else torch.bfloat16
    if kind == "prologue":
        ins = [r(B, T, Hk, D), r(B, T, Hk, D), r(B, T, Hv, D), r(B, T, Hv), r(B, T, Hv)]
        ins = [t.to(dt) for t in ins] + [r(Hv), r(Hv)]
        call = gdn.gated_delta_prologue
    else:
        q, k = (F.normalize(r(B, T, Hk, D), dim=-1).to(dt) for _ in range(2))
        ins = [q, k, r(B, T, Hv, D).to(dt), -F.softplus(r(B, T, Hv)), torch.sigmoid(r(B, T, Hv)).to(dt)]
        call = lambda *a: gdn.gated_delta_trainable(*a, log_decay=True)  # noqa: E731
    ins.append(0.1 * r(B, Hv, D, D) if carried else None)
    leaves = [t.requires_grad_(True) for t in ins if t is not None]
    y, s = call(*ins)
    dy, ds = torch.randn(y.shape, device="cuda", generator=gen).to(y.dtype), r(*s.shape)
    for outs, cots, full in (((y,), (dy,), (dy, torch.zeros_like(s))), ((s,), (ds,), (torch.zeros_like(y), ds))):
        one = torch.autograd.grad(outs, leaves, cots, retain_graph=True)
        both = torch.autograd.grad((y, s), leaves, full, retain_graph=True)
        assert all(a.dtype == x.dtype and torch.equal(a, b) for a, b, x in zip(one, both, leaves))
    assert all(bool(g.isfinite().all()) for g in one)

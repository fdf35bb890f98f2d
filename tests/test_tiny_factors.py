"""dL/dg at tiny decay factors where more (chunk, value head) pairs hold one than the device has CUs, so that the
blocks of the exact replay each take several of the listed pairs, and where none does, so that the list is empty; and
with no tokens, where the workspace that holds the list has no bytes.
Against the oracle, within the 2e-3 of each output's largest value that the other tests of bf16 inputs allow (one
rounding of the inputs, hi/lo products)."""
import numpy as np
import pytest

from helpers import normwise, small_case
from quotebound_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("every", [64, 0], ids=["one in each pair", "none"])
def test_listed_pairs(oracle, every):
    import torch

    from quotebound_amd import gdn
    from quotebound_amd.synthetic import round_bf16

    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    B, T, Hk, Hv, Dv = 1, 64 * 33 + 5, 4, 8, 32  # 34 chunks of 8 heads: 272 pairs on 256 CUs
    inp = small_case(B, T, Hk, Hv, 128, Dv, seed=12, log_decay=False)
    inp["g"] = np.clip(inp["g"], 2.0 ** -9, None)
    if every:
        inp["g"][0, 3::every] = np.float32(2.0 ** -14)
        inp["g"][0, 4::4 * every] = 0.0
    for n in ("q", "k", "v", "beta", "dy"):
        inp[n] = round_bf16(np.asarray(inp[n], np.float32)).reshape(inp[n].shape)
    inp = {n: np.asarray(x, np.float32) for n, x in inp.items()}
    five = [inp[n] for n in ("q", "k", "v", "g", "beta")]
    _, _, ck = oracle.fwd(*five, inp["s0"], g_is_log=False, dtype=np.float32)
    exp = oracle.bwd(*five, ck, inp["dy"], inp["ds_out"], g_is_log=False, dtype=np.float32)
    d = {n: torch.tensor(x).cuda() for n, x in inp.items()}
    for n in ("q", "k", "v", "beta"):
        d[n] = d[n].bfloat16()
    dev = [d[n] for n in ("q", "k", "v", "g", "beta")]
    _, _, ckpt = gdn.forward(*dev, d["s0"], design=_lib.CHUNKED, out_f32=True)
    got = gdn.backward(*dev, ckpt, d["dy"], d["ds_out"], design=_lib.CHUNKED, out_f32=True)
    again = gdn.backward(*dev, ckpt, d["dy"], d["ds_out"], design=_lib.CHUNKED, out_f32=True)
    torch.cuda.synchronize()
    for name, x, y, e in zip(("dq", "dk", "dv", "dg", "dbeta", "ds0"), got, again, exp):
        assert torch.equal(x, y), name
        assert normwise(x.cpu().numpy(), e) <= 2e-3, (name, normwise(x.cpu().numpy(), e))


@pytest.mark.parametrize("cu", [None, [0, 0, 0, 0]], ids=["batch", "packed"])
@pytest.mark.parametrize("design", [_lib.CHUNKED, _lib.RECURRENT], ids=["chunked", "recurrent"])
def test_no_tokens_leave_the_workspace_alone(design, cu):
    """T = 0 asks for 0 bytes of workspace: whatever the pointer points at stays as it was, forward and backward, and
    the final state is S0 and dS0 its cotangent."""
    import torch

    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    B, N, Hk, Hv, D = (3 if cu is None else 1), 3, 2, 4, 128
    desc, keep = _lib.make_desc(B, 0, Hk, Hv, D, D, dtype=_lib.BF16, g_is_log=False, design=design, cu_seqlens=cu)
    assert _lib.validate(desc) is None and _lib.workspace_bytes(desc) == 0
    s0, ds_out = torch.randn(N, Hv, D, D, device="cuda"), torch.randn(N, Hv, D, D, device="cuda")
    s_out, ds0 = torch.empty_like(s0), torch.empty_like(s0)
    other = torch.full((256,), 0x5A, dtype=torch.uint8, device="cuda")
    p, none, stream = (lambda t: t.data_ptr()), [None] * 5, torch.cuda.current_stream().cuda_stream
    _lib.fwd(desc, *none, p(s0), None, p(s_out), None, p(other), stream)
    _lib.bwd(desc, *none, None, None, p(ds_out), *none, p(ds0), p(other), stream)
    torch.cuda.synchronize()
    assert torch.equal(s_out, s0) and torch.equal(ds0, ds_out)
    assert bool((other == 0x5A).all())

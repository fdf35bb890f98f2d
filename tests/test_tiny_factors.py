"""dL/dg at tiny decay factors where more (chunk, value head) pairs hold one than the device has CUs, so that the
blocks of the exact replay each take several of the listed pairs, and where none does, so that the list is empty.
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

"""The float32 chunk kernels (design 1 on float32 inputs at Dk = 128, sequences of 160 steps and more forward, 192
backward) against the oracle, on the GPU through the Python entry points, at the sizes where they can go wrong: the
shortest sequences that take them and the ones around whole chunks, one to three value heads per key head, one and several row blocks, ragged
packed batches with empty sequences, the decay as log and as factor (negative and zero factors among them), and values
that are not finite, which must reach the outputs that they reach step by step and no others.

Tolerance: 1e-5 of each output's largest value, the float32 criterion of the other tests. (The sums run over at most
128 terms of float32 products, 16 at a time: about 2e-7 of the values' size.)
"""
import numpy as np
import pytest

from helpers import GRAD_NAMES, normwise, small_case
from quotebound_amd import _lib

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.fixture(scope="module")
def torch_dev():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    _lib.load()
    return torch


def _run(torch, inp, cu=None, log_decay=True):
    from quotebound_amd import gdn

    d = {n: None if x is None else torch.tensor(np.asarray(x, np.float32)).cuda() for n, x in inp.items()}
    five = (d["q"], d["k"], d["v"], d["g"], d["beta"])
    y, s_out, ckpt = gdn.forward(*five, d["s0"], log_decay=log_decay, cu_seqlens=cu)
    y2, s2, _ = gdn.forward(*five, d["s0"], log_decay=log_decay, cu_seqlens=cu, save_ckpt=False)
    grads = gdn.backward(*five, ckpt, d["dy"], d["ds_out"], log_decay=log_decay, cu_seqlens=cu)
    torch.cuda.synchronize()
    assert torch.equal(y.isnan(), y2.isnan()) and torch.equal(y.nan_to_num(), y2.nan_to_num())
    assert torch.equal(s_out.nan_to_num(), s2.nan_to_num())
    return dict(zip(("y", "s_out") + GRAD_NAMES, [t.cpu().numpy() for t in (y, s_out, *grads)]))


def _check(got, exp, names=("y", "s_out") + GRAD_NAMES):
    for n in names:
        bad = np.isfinite(exp[n])
        assert np.array_equal(np.isfinite(got[n]), bad), n
        err = normwise(np.where(bad, got[n], 0.0), np.where(bad, exp[n], 0.0))
        assert err <= TOL, (n, err)


def _float32(inp):
    return {n: None if x is None else np.asarray(x, np.float32) for n, x in inp.items()}


@pytest.mark.parametrize("B,T,Hk,Hv,Dv,carried", [
    (1, 159, 2, 4, 128, True),   # one step too short for either
    (1, 160, 2, 4, 128, True),   # the forward alone
    (2, 192, 1, 1, 32, False),   # both; whole chunks, one value head per key head, one block of state rows
    (1, 193, 1, 3, 96, True),    # one step into the fourth chunk, three heads per key head, an odd count of row blocks
    (3, 255, 2, 2, 64, True),
    (1, 1037, 16, 32, 128, True),
])
def test_shapes(torch_dev, oracle, B, T, Hk, Hv, Dv, carried):
    inp = _float32(small_case(B, T, Hk, Hv, 128, Dv, seed=T, s0=carried, ds_out=carried))
    _check(_run(torch_dev, inp), oracle.fwd_bwd(inp, dtype=np.float32))


def test_packed(torch_dev, oracle):
    lens = [192, 0, 5, 64, 300, 1, 129]
    T, N, Hk, Hv = sum(lens), len(lens), 2, 4
    inp = small_case(1, T, Hk, Hv, 128, 64, seed=5)
    r = np.random.default_rng(6)
    inp["s0"], inp["ds_out"] = r.normal(0.0, 0.1, (N, Hv, 64, 128)), r.standard_normal((N, Hv, 64, 128))
    inp, cu = _float32(inp), np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    got = _run(torch_dev, inp, cu)
    _check(got, oracle.fwd_bwd(inp, cu_seqlens=cu, dtype=np.float32))
    assert np.array_equal(got["s_out"][1], inp["s0"][1]) and np.array_equal(got["ds0"][1], inp["ds_out"][1])


def test_decay_factors(torch_dev, oracle):
    """Factors of either sign and zero: the forward runs on their logs with the sign apart."""
    inp = _float32(small_case(1, 200, 2, 4, 128, 64, seed=8, log_decay=False))
    inp["g"][0, ::7] *= -1.0
    inp["g"][0, 50] = 0.0
    inp["g"][0, 130, 1] = 1e-30
    y, s_out, _ = oracle.fwd(*(inp[n] for n in ("q", "k", "v", "g", "beta", "s0")), g_is_log=False, dtype=np.float32)
    _check(_run(torch_dev, inp, log_decay=False), {"y": np.asarray(y), "s_out": np.asarray(s_out)}, ("y", "s_out"))


@pytest.mark.parametrize("where", ["v", "dy", "log_decay"])
def test_not_finite(torch_dev, oracle, where):
    """A NaN in v reaches y and the state from its step on and its row only, one in dy the gradients up to its step; a
    log-decay of -inf is a factor of 0 and reaches nothing."""
    inp = _float32(small_case(1, 200, 2, 4, 128, 64, seed=9))
    if where == "v":
        inp["v"][0, 100, 2, 17] = np.nan
    elif where == "dy":
        inp["dy"][0, 100, 2, 17] = np.nan
    else:
        inp["g"][0, 100, 2] = -np.inf
    got = _run(torch_dev, inp)
    if where == "log_decay":
        exp = oracle.fwd_bwd(inp, dtype=np.float32)
        _check(got, exp, ("y", "s_out", "dq", "dk", "dv", "dbeta", "ds0"))
        return
    clean = _run(torch_dev, dict(inp, **{where: np.nan_to_num(inp[where])}))
    if where == "v":
        bad = np.zeros(inp["v"].shape, bool)
        bad[0, 100:, 2, 17] = True
        assert np.array_equal(np.isnan(got["y"]), bad)
        assert np.isnan(got["s_out"][0, 2, 17]).all() and np.isnan(got["s_out"]).sum() == 128
        assert normwise(got["y"][~bad], clean["y"][~bad]) <= TOL
    else:
        bad = np.zeros(inp["v"].shape, bool)
        bad[0, :101, 2, 17] = True
        assert np.array_equal(np.isnan(got["dv"]), bad)
        assert not np.isnan(got["y"]).any() and not np.isnan(got["dq"][0, 101:]).any()
        assert np.isnan(got["ds0"][0, 2, 17]).all() and np.isnan(got["ds0"]).sum() == 128
        assert normwise(got["dv"][~bad], clean["dv"][~bad]) <= TOL


def _device(torch, inp):
    return {n: torch.tensor(x).cuda() for n, x in inp.items()}


def test_element_alignment(torch_dev):
    """v, g, beta, dy and the states need only their elements' alignment: one float past a 16-byte boundary gives the
    same bits."""
    torch = torch_dev
    from quotebound_amd import gdn

    d = _device(torch, _float32(small_case(1, 200, 2, 4, 128, 64, seed=10)))

    def off(t):
        x = torch.empty(t.numel() + 1, device="cuda")[1:].view(t.shape)
        return x.copy_(t)

    def both(d):
        five = (d["q"], d["k"], d["v"], d["g"], d["beta"])
        y, s_out, ckpt = gdn.forward(*five, d["s0"], log_decay=True)
        return [y, s_out, *gdn.backward(*five, ckpt, d["dy"], d["ds_out"], log_decay=True)]

    moved = {n: t if n in ("q", "k") else off(t) for n, t in d.items()}
    assert all(moved[n].data_ptr() % 16 == 4 for n in ("v", "g", "beta", "dy", "s0", "ds_out"))
    assert all(torch.equal(x, y) for x, y in zip(both(d), both(moved)))


def test_in_a_graph(torch_dev):
    """Captured in a HIP graph: replays on new inputs give the eager call's bits, with eager work between them, and a
    value that is not finite raises the flag in the replay that has it and in no other."""
    torch = torch_dev
    from quotebound_amd import gdn

    def call(d):
        five = (d["q"], d["k"], d["v"], d["g"], d["beta"])
        y, s_out, ckpt = gdn.forward(*five, d["s0"], log_decay=True)
        return [y, s_out, *gdn.backward(*five, ckpt, d["dy"], d["ds_out"], log_decay=True)]

    cases = [_device(torch, _float32(small_case(1, 200, 2, 4, 128, 64, seed=s))) for s in (20, 21, 22)]
    cases[1]["v"][0, 150, 1, 3] = float("nan")
    static = {n: t.clone() for n, t in cases[0].items()}
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(static)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call(static)
    for c in (cases[0], cases[1], cases[2], cases[0]):
        want = call(c)
        for n, t in static.items():
            t.copy_(c[n])
        graph.replay()
        torch.cuda.synchronize()
        for x, y in zip(out, want):
            assert torch.equal(x.isnan(), y.isnan()) and torch.equal(x.nan_to_num(), y.nan_to_num())

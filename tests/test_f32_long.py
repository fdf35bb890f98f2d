"""The recurrent design on long float32 sequences against the oracle, on the GPU through the Python and the C entry
points: lengths around whole chunks, one to three value heads per key head, one and several row blocks, ragged packed
batches with empty sequences, the decay as log and as factor (negative and zero factors among them), values that are not
finite, which must reach the outputs that they reach step by step and no others; and what the step-by-step order
promises at any length: the float32 oracle's accuracy on keys that are nearly parallel, the same bits as the per-token
states and as one-token calls, the same bits for a sequence alone and packed with others, and states updated in place
(these in the chunked design too).

Tolerance, where no other is derived: 1e-5 of each output's largest value, the float32 criterion of the other tests.
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
    (1, 159, 2, 4, 128, True),
    (1, 160, 2, 4, 128, True),
    (2, 192, 1, 1, 32, False),   # whole chunks, one value head per key head, two blocks of state rows
    (1, 193, 1, 3, 96, True),    # one step into the fourth chunk, three heads per key head
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
    """Factors of either sign, tiny and zero."""
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
        _check(got, exp)
        assert (got["dg"][0, 100, 2] == 0.0).all()  # exp(-inf) times the state's inner product
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
    """Captured in a HIP graph: replays on new inputs give the eager call's bits, with eager work between them, a
    value that is not finite in one of them included."""
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


# ---- what the step-by-step order promises at any length --------------------------------------------------------------


def _near_parallel(T, spread, seed):
    """Keys with a common direction, `spread` times a random one added: the 64 x 64 systems of a chunkwise form are then
    badly conditioned, while the step-by-step form does not meet them."""
    inp = small_case(1, T, 1, 2, 128, 64, seed=seed)
    r = np.random.default_rng(seed + 1)
    k = r.standard_normal((1, 1, 1, 128)) / np.sqrt(128) + spread * r.standard_normal((1, T, 1, 128)) / np.sqrt(128)
    inp["k"] = k / np.linalg.norm(k, axis=-1, keepdims=True)
    return inp


@pytest.mark.parametrize("spread,beta,decay", [(None, None, None), (0.3, 1.0, 0.0), (0.1, 1.9, 0.0), (0.3, 2.2, 0.05)])
def test_accuracy_of_the_step_by_step_form(torch_dev, oracle, spread, beta, decay):
    """No further from the 64-bit oracle than twice the float32 oracle, output by output in the 2-norm: the same steps
    with the same roundings, the sums over a row in another order. (spread None: small_case's independent keys.)"""
    T = 512
    inp = small_case(1, T, 1, 2, 128, 64, seed=30) if spread is None else _near_parallel(T, spread, 31)
    if spread is not None:
        inp["beta"], inp["g"] = np.full((1, T, 2), beta), np.full((1, T, 2), -decay)
    inp = _float32(inp)
    exact, plain = oracle.fwd_bwd(inp, dtype=np.float64), oracle.fwd_bwd(inp, dtype=np.float32)
    got = _run(torch_dev, inp)
    err = lambda x, n: np.linalg.norm(x[n].astype(np.float64) - exact[n]) / np.linalg.norm(exact[n])  # noqa: E731
    errs = {n: (float(err(got, n)), float(err(plain, n))) for n in ("y", "s_out") + GRAD_NAMES}
    print(f"spread {spread} beta {beta} decay {decay}:", {n: f"{g:.1e} ({o:.1e})" for n, (g, o) in errs.items()})
    assert all(g <= 2.0 * o for g, o in errs.values()), errs


def test_bits_of_the_per_token_states(torch_dev):
    """The forward, the forward that keeps the state after every token, and one-token calls agree bit for bit, whatever
    the length: a decoder may take a prompt in one call and roll back to any token of it."""
    torch = torch_dev
    from quotebound_amd import gdn

    d = _device(torch, _float32(small_case(1, 300, 2, 4, 128, 64, seed=40)))
    five = [d[n] for n in ("q", "k", "v", "g", "beta")]
    y, s_out, _ = gdn.forward(*five, d["s0"], log_decay=True)
    y_rows, rows = gdn.forward_rows(*five, d["s0"], log_decay=True)
    assert torch.equal(y, y_rows) and torch.equal(s_out, rows[:, -1])
    state = rows[:, 249].contiguous()
    for t in range(250, 300):
        y_t, state = gdn.gated_delta(*(x[:, t:t + 1] for x in five), state, log_decay=True)
        assert torch.equal(y_t, y[:, t:t + 1]), t
    assert torch.equal(state, s_out)


def test_bits_of_a_packed_sequence(torch_dev):
    """A sequence's results do not depend on what it is packed with: the bits of a call of its own, forward and
    backward."""
    torch = torch_dev
    from quotebound_amd import gdn

    lens = [70, 260, 0, 5]
    cu = [0] + [int(x) for x in np.cumsum(lens)]
    inp = small_case(1, sum(lens), 2, 4, 128, 64, seed=41)
    r = np.random.default_rng(42)
    inp["s0"], inp["ds_out"] = r.normal(0.0, 0.1, (4, 4, 64, 128)), r.standard_normal((4, 4, 64, 128))
    d = _device(torch, _float32(inp))

    def call(x, s0, dy, ds, **kw):
        y, s_out, ckpt = gdn.forward(*x, s0, log_decay=True, **kw)
        dq, dk, dv, dg, db, ds0 = gdn.backward(*x, ckpt, dy, ds, log_decay=True, **kw)
        return (y, dq, dk, dv, dg, db), (s_out, ds0)

    five = [d[n] for n in ("q", "k", "v", "g", "beta")]
    tokens, states = call(five, d["s0"], d["dy"], d["ds_out"], cu_seqlens=cu)
    for i, n in enumerate(lens):
        own = slice(cu[i], cu[i + 1])
        t1, s1 = call([x[:, own] for x in five], d["s0"][i:i + 1], d["dy"][:, own], d["ds_out"][i:i + 1])
        assert all(torch.equal(x[:, own], z) for x, z in zip(tokens, t1)), (i, n)
        assert all(torch.equal(x[i:i + 1], z) for x, z in zip(states, s1)), (i, n)


@pytest.mark.parametrize("design,where", [(_lib.RECURRENT, w) for w in (None, "v", "k", "beta", "s0", "dy", "ds_out")] +
                         [(_lib.CHUNKED, None), (_lib.CHUNKED, "v")])
def test_states_in_place(torch_dev, design, where):
    """Through the C entry points: s_out in s0's buffer and ds0 in ds_out's give what separate buffers give, with all
    values finite and with a NaN in one of the inputs. (The chunked design on bf16 activations.)"""
    torch = torch_dev
    T, Hk, Hv, Dv = 200, 2, 4, 64
    d = _device(torch, _float32(small_case(1, T, Hk, Hv, 128, Dv, seed=43)))
    if where:
        d[where].view(-1)[d[where].numel() // 2 + 17] = float("nan")
    if design == _lib.CHUNKED:
        d.update({n: d[n].bfloat16() for n in ("q", "k", "v", "beta", "dy")})
    dtype = _lib.F32 if design == _lib.RECURRENT else _lib.BF16
    desc, keep = _lib.make_desc(1, T, Hk, Hv, 128, Dv, dtype=dtype, design=design)
    stream = torch.cuda.current_stream().cuda_stream

    def call(in_place):
        x = {n: t.clone() for n, t in d.items()}
        out = {n: torch.empty_like(x[m]) for n, m in (("y", "v"), ("dq", "q"), ("dk", "k"), ("dv", "v"), ("dg", "g"),
                                                      ("dbeta", "beta"))}
        out["s_out"], out["ds0"] = (x["s0"], x["ds_out"]) if in_place else (x["s0"].clone(), x["ds_out"].clone())
        ckpt = torch.empty(_lib.ckpt_bytes(desc) // 4, device="cuda")
        ws = torch.empty(_lib.workspace_bytes(desc), dtype=torch.uint8, device="cuda")
        p = lambda *names: [(x.get(n) if n in x else out[n]).data_ptr() for n in names]  # noqa: E731
        _lib.fwd(desc, *p("q", "k", "v", "g", "beta", "s0", "y", "s_out"), ckpt.data_ptr(), ws.data_ptr(), stream)
        _lib.bwd(desc, *p("q", "k", "v", "g", "beta"), ckpt.data_ptr(),
                 *p("dy", "ds_out", "dq", "dk", "dv", "dg", "dbeta", "ds0"), ws.data_ptr(), stream)
        torch.cuda.synchronize()
        return out

    apart, together = call(False), call(True)
    for n in apart:
        assert torch.equal(apart[n].isnan(), together[n].isnan()), n
        assert torch.equal(apart[n].nan_to_num(), together[n].nan_to_num()), n
    if where is None:
        assert all(bool(t.isfinite().all()) for t in apart.values())

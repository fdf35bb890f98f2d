"""What the recurrent design asks for and refuses, without a GPU: its workspace is the partials of the backward's row
blocks and nothing more, on float32 as on bf16, and the backward without a workspace takes every call whose partials fit
its static array and none beyond."""
import pytest

from quotebound_amd import _lib


def _partials(T, Hv, Dk, Dv):
    rows = 16 if Dk <= 128 else 8
    nblk = -(-Dv // rows)
    return (2 * T * Hv * nblk * Dk + 2 * T * Hv * nblk) * 4


@pytest.mark.parametrize("kw", [
    dict(T=160), dict(T=159), dict(T=4096, dtype=_lib.BF16), dict(T=4096, Dk=64), dict(T=4096, Dv=48),
    dict(T=160, g_is_log=False), dict(T=4096, cu_seqlens=[0, 100, 200, 4096]), dict(T=0),
    dict(T=360, cu_seqlens=list(range(201)) + [360]),
])
def test_workspace_is_the_partials(kw):
    d = dict(B=1, Hk=2, Hv=4, Dk=128, Dv=128, dtype=_lib.F32, design=_lib.RECURRENT)
    d.update(kw)
    desc, keep = _lib.make_desc(**d)
    assert _lib.validate(desc) is None
    assert _lib.workspace_bytes(desc) == _partials(d["T"], d["Hv"], d["Dk"], d["Dv"])


def test_static_scratch_limit():
    """The largest T whose partials fit the static array gets as far as its pointers, the next is refused."""
    T = _lib.STATIC_SCRATCH_BYTES // _partials(1, 4, 128, 128)
    for n, why in ((T, "ckpt is null"), (T + 1, "without allocation needs")):
        desc, _ = _lib.make_desc(1, n, 2, 4, 128, 128, dtype=_lib.F32, design=_lib.RECURRENT)
        with pytest.raises(RuntimeError, match=why):
            _lib.bwd_static(desc, 16, 16, 16, 16, 16, None, 16, None, 16, 16, 16, 16, 16, None, None)

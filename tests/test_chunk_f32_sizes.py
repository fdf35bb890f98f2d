"""Which calls the float32 chunk kernels take, seen from the workspace a call asks for (16 bytes for their flag after the
recurrent design's partials where they may run), and that what the backward without a workspace accepts has not
changed by those bytes. No GPU."""
import pytest

from quotebound_amd import _lib


def _partials(T, Hv, Dk, Dv):
    rows = 16 if Dk <= 128 else 8
    nblk = -(-Dv // rows)
    return (2 * T * Hv * nblk * Dk + 2 * T * Hv * nblk) * 4


@pytest.mark.parametrize("kw,flag", [
    (dict(T=160), 16),
    (dict(T=159), 0),                                   # too short
    (dict(T=160, g_is_log=False), 16),
    (dict(T=4096, dtype=_lib.BF16), 0),                 # float32 only
    (dict(T=4096, Dk=64), 0),                           # keys of 128 only
    (dict(T=4096, Dv=48), 0),                           # state rows in blocks of 32
    (dict(T=4096, cu_seqlens=[0, 100, 200, 4096]), 16),  # the longest sequence counts
    (dict(T=320, cu_seqlens=[0, 100, 200, 320]), 0),
    (dict(T=4000 + 160, cu_seqlens=[i for i in range(0, 251)] + [4160]), 16),
    (dict(T=200 + 160, cu_seqlens=[i for i in range(0, 201)] + [360]), 0),  # their intermediates would not fit
    (dict(T=256, Hk=16, Hv=131072), 0),                 # offsets past 32 bits
])
def test_flag_bytes(kw, flag):
    d = dict(B=1, Hk=2, Hv=4, Dk=128, Dv=128, dtype=_lib.F32, design=_lib.RECURRENT)
    d.update(kw)
    desc, keep = _lib.make_desc(**d)
    assert _lib.validate(desc) is None
    assert _lib.workspace_bytes(desc) == _partials(d["T"], d["Hv"], d["Dk"], d["Dv"]) + flag


def test_static_scratch_limit_counts_the_partials_alone():
    """The largest T whose partials fit the static array is accepted as before (it gets as far as its pointers)."""
    T = _lib.STATIC_SCRATCH_BYTES // _partials(1, 4, 128, 128)
    for n, why in ((T, "ckpt is null"), (T + 1, "without allocation needs")):
        desc, _ = _lib.make_desc(1, n, 2, 4, 128, 128, dtype=_lib.F32, design=_lib.RECURRENT)
        with pytest.raises(RuntimeError, match=why):
            _lib.bwd_static(desc, 16, 16, 16, 16, 16, None, 16, None, 16, 16, 16, 16, 16, None, None)

"""The plans that calls of one shape share (a descriptor and its sizes, no tensor): found again by their values, the
least recently used ones dropped, and a refused call refused each time."""
import pytest

from quotebound_amd import _lib


def _make(T):
    desc, keep = _lib.make_desc(1, T, 2, 4, 128, 128)
    return _lib.Plan(desc, keep, _lib.workspace_bytes(desc), _lib.ckpt_bytes(desc) // 4)


@pytest.fixture
def plans():
    kept = dict(_lib._plans)
    _lib._plans.clear()
    yield _lib._plans
    _lib._plans.clear()
    _lib._plans.update(kept)


def test_same_values_same_plan(plans):
    a = _lib.plan(("a", 64), lambda: _make(64))
    assert _lib.plan(("a", 64), lambda: pytest.fail("formed again")) is a
    b = _lib.plan(("a", 65), lambda: _make(65))
    assert b is not a and b.desc.T == 65
    assert (b.workspace, b.ckpt_floats) == (_lib.workspace_bytes(b.desc), _lib.ckpt_bytes(b.desc) // 4)


def test_bounded_by_last_use(plans):
    first = _lib.plan(0, lambda: _make(64))
    for i in range(1, _lib._PLANS_KEPT):
        _lib.plan(i, lambda: _make(64))
    assert _lib.plan(0, lambda: pytest.fail("dropped")) is first
    _lib.plan(_lib._PLANS_KEPT, lambda: _make(64))
    assert len(plans) == _lib._PLANS_KEPT and 0 in plans and 1 not in plans


def test_refusals_are_not_kept(plans):
    def refuse():
        raise RuntimeError("no")

    for _ in range(2):
        with pytest.raises(RuntimeError, match="no"):
            _lib.plan("bad", refuse)
    assert "bad" not in plans

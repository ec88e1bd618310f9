"""Launch plans on the CPU: what is recorded and replayed, with a stand-in for the library that notes the addresses it is given."""
import struct

import pytest
import torch

from fastfold_amd import _lib, _plan


class _Library:
    """Notes the buffer of every ``ffk_fill_zero``, launched by itself or out of a plan."""

    def __init__(self):
        self.seen, self.replays = [], 0

    def ffk_fill_zero(self, p, nbytes, stream):
        self.seen.append(p)
        return 0

    def ffk_run_plan(self, blob, size, bases, n, stream):
        self.replays += 1
        at = 0
        while at < size:
            code, slots, relocs, _ = struct.unpack_from("<iiii", blob, at)
            assert _plan.OPS[code] == "ffk_fill_zero"
            args = list(struct.unpack_from("<%dQ" % slots, blob, at + 16 + 16 * relocs))
            for k in range(relocs):
                slot, base, off = struct.unpack_from("<iiq", blob, at + 16 + 16 * k)
                args[slot] = bases[base] + off
            self.seen.append(args[0])
            at += 16 + 16 * relocs + 8 * slots
        return 0


@pytest.fixture
def library(monkeypatch):
    lib = _Library()
    monkeypatch.setattr(_lib, "load", lambda path=None: lib)
    monkeypatch.setattr(_lib, "stream_ptr", lambda: 0)
    return lib


def _call(lib, owner, tensors, key="k"):
    """One call whose sequence launches on every tensor; the addresses it launched on."""
    lib.seen = []
    _plan.run(owner, key, tensors, lambda: [_lib.fill_zero(t) for t in tensors if t is not None])
    return lib.seen


def _ptrs(tensors):
    return [t.data_ptr() for t in tensors if t is not None]


@pytest.mark.parametrize("form", ["one", "overlap", "optional"])
def test_a_plan_recorded_with_shared_buffers_serves_no_others(library, form):
    owner = torch.nn.Linear(2, 2)
    x, a, b, big = torch.zeros(8), torch.zeros(8), torch.zeros(8), torch.zeros(16)
    shared = {"one": [x, a, a], "overlap": [x, big[:8], big[4:12]], "optional": [x, None, x]}[form]
    other = {"one": [x, a, b], "overlap": [x, big[:8], big[8:]], "optional": [x, None, b]}[form]
    for tensors in (shared, other, shared, other, other[::-1], shared):
        assert _call(library, owner, tensors) == _ptrs(tensors)
    assert library.replays == 4                # all but the first call of each pattern (the reversed one has that of ``other``)
    for tensors in ([a, b, a, b], [b, a, b, a], [x, a, x, a]):         # one pattern, whichever buffer lies first in memory
        assert _call(library, owner, tensors, "pairs") == _ptrs(tensors)
    assert library.replays == 6


def test_the_plan_dropped_is_the_one_used_longest_ago(library):
    owner, x = torch.nn.Linear(2, 2), torch.zeros(8)
    for k in range(_plan._MAX_PLANS):
        _call(library, owner, [x], k)
    for k in range(_plan._MAX_PLANS, _plan._MAX_PLANS + 4):
        _call(library, owner, [x], 0)                 # used in between
        _call(library, owner, [x], k)
    assert library.replays == 4
    plans = owner.__dict__["_plan_state"].plans
    assert [k[0] for k in plans] == [*range(5, _plan._MAX_PLANS + 3), 0, _plan._MAX_PLANS + 3]


def test_values_derived_from_a_mask_without_a_version_counter():
    """Tensors made under ``torch.inference_mode`` have none: built once per mask inside a cache, like the others."""
    from fastfold_amd.model.fastnn import _fused as F_
    with torch.inference_mode():
        masks = [torch.ones(4, 4), torch.ones(4, 4)]
        masks.append(masks[0].t())
        with F_.mask_cache():
            got = [F_._mask_derived(m, "twice", lambda m=m: 2 * m) for m in masks + masks]
    assert all(got[i] is got[i + 3] for i in range(3)) and len({id(t) for t in got}) == 3

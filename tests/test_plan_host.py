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

"""Launch plans: the launches of a block, recorded once per shape from the Python sequence that issues them and replayed
by the library (``ffk_run_plan``) with the buffers of each call.

The sequences of ``model/fastnn/_fused.py`` prepare every launch in Python - descriptors, packed weights, scratch tensors,
the foreign call - at about 20 microseconds of host time each, 0.57 ms for a block of 25 launches, while the GPU needs 5 to
30 microseconds for one up to N_res = 256.  ``run`` records such a sequence while it executes (nothing is executed twice)
and from then on replays it: the 48-block trunk at N_seq = 128, N_res = 77 went from 30.6 to 4.6 ms of host time.

A plan holds no results.  Every pointer of a recorded launch is one of
  * a caller's buffer (activations, masks and what is derived from them), patched on each replay - of calls in which the same
    buffers coincide as in the recorded one,
  * scratch, laid out in one allocation that each replay makes for itself on its own stream,
  * a packed weight or parameter, which the plan keeps alive; a plan is dropped as soon as a parameter of its module has
    changed (another tensor, or another version of it), exactly as the packed weights are.
A sequence that issues anything else is not planned and keeps running in Python.
"""
import ctypes
import struct
import threading
from collections import OrderedDict

import torch

from . import _lib

OPS = ["ffk_fused_linear", "ffk_bgemm_nt", "ffk_attention_fwd", "ffk_pair_bias", "ffk_opm_fused", "ffk_transition_fused",
       "ffk_gated_out_fused", "ffk_global_attention_core", "ffk_layernorm_fwd", "ffk_fill_zero", "ffk_attention_fwd_lse",
       "ffk_attention_bwd_rows", "ffk_transpose_batched", "ffk_weight_grad", "ffk_layernorm_bwd_rows", "ffk_scale_rows",
       "ffk_att_gate_bwd", "ffk_trimul_gate_bwd", "ffk_glu_bwd", "ffk_bias_cols", "ffk_slice_sum",
       "ffk_attention_block", "ffk_attention_heads", "ffk_transition_block"]   # order of FFK_OP_*
_CODE = {name: i for i, name in enumerate(OPS)}
_MAX_PLANS = 16               # per module: shapes in use at a time
_ALIGN = 512                  # of scratch buffers, as torch's allocator aligns its blocks
# Large buffers begin 4 KB further into a 2 MB page each: operands of one launch that all begin on a page boundary share
# their memory channels (4 extra-MSA blocks at 1024 x 384: 8.16 ms against 8.22 on page boundaries, 8.26 packed tightly).
_LARGE, _PAGE, _STAGGER = 1 << 20, 1 << 21, 1 << 12

builds = 0                    # counts packed-weight (and scratch-operand) builds: a recording that saw one is not kept


epoch = 0                     # counts explicit invalidations of packed weights: every plan of before is void


def note_build():
    global builds
    builds += 1


def invalidate():
    global epoch
    epoch += 1


class _NotPlannable(Exception):
    pass


def _pointer_slots(struct_type, base=0):
    """Slot numbers (8-byte words) of the pointer fields of a ctypes structure, arrays of structures included."""
    out = []
    for name, typ in struct_type._fields_:
        off = base + getattr(struct_type, name).offset
        if typ is ctypes.c_void_p:
            out.append(off // 8)
        elif isinstance(typ, type) and issubclass(typ, ctypes.Array) and issubclass(typ._type_, ctypes.Structure):
            for i in range(typ._length_):
                out += _pointer_slots(typ._type_, off + i * ctypes.sizeof(typ._type_))
    return out


_DESC_POINTERS = {}


class _Recorder:
    """Turns the launches of one execution into a plan.  ``tensors``: the caller's buffers, in the order replays pass them."""

    def __init__(self, tensors, keep):
        self.bound = [(t.data_ptr(), t.data_ptr() + t.numel() * t.element_size(), i + 2) for i, t in enumerate(tensors)
                      if t is not None]
        self.keep = [(t.data_ptr(), t.data_ptr() + t.numel() * t.element_size()) for t in keep]
        self.temps, self.held = [], []
        self.bump = self.peak = self.floor = 0
        self.out = []
        self.failed = None

    def alloc(self, t):
        used = t.numel() * t.element_size()
        size = -(-used // _ALIGN) * _ALIGN if used < _LARGE else -(-used // _PAGE) * _PAGE + _STAGGER
        self.temps.append((t.data_ptr(), t.data_ptr() + used, self.bump))
        self.bump += size
        self.peak = max(self.peak, self.bump)

    def scope(self):
        """A sub-module begins: the scratch of the one before is dead."""
        self.temps = list(self.held)
        self.bump = self.floor

    def hold(self):
        """What has been allocated so far stays alive until the end of the sequence."""
        self.held = list(self.temps)
        self.floor = self.bump

    def _reloc(self, p):
        for lo, hi, off in reversed(self.temps):       # the youngest first: memory freed in between may have been reused
            if lo <= p < hi:
                return 1, off + p - lo
        for lo, hi, i in self.bound:
            if lo <= p < hi:
                return i, p - lo
        if any(lo <= p < hi for lo, hi in self.keep):
            return 0, p
        raise _NotPlannable("a launch uses a buffer the plan does not know")

    def note(self, name, args):
        if self.failed is not None:
            return
        try:
            code = _CODE.get(name)
            if code is None:
                raise _NotPlannable("%s cannot be replayed" % name)
            args = args[:-1]
            relocs = []
            if len(args) == 1:                          # a descriptor
                d = args[0]._obj
                slots = bytearray(bytes(d))
                ptrs = _DESC_POINTERS.get(type(d))
                if ptrs is None:
                    ptrs = _DESC_POINTERS[type(d)] = _pointer_slots(type(d))
            else:
                slots, ptrs = bytearray(), []
                for i, (a, typ) in enumerate(zip(args, _lib.SIGNATURES[name])):
                    if typ is ctypes.c_void_p:
                        ptrs.append(i)
                        slots += struct.pack("<Q", a or 0)
                    elif typ is ctypes.c_float:
                        slots += struct.pack("<fI", a, 0)
                    else:
                        slots += struct.pack("<q", a)
            for i in ptrs:
                p = struct.unpack_from("<Q", slots, 8 * i)[0]
                if p:
                    base, off = self._reloc(p)
                    if base:
                        relocs.append(struct.pack("<iiq", i, base, off))
            self.out.append(struct.pack("<iiii", code, len(slots) // 8, len(relocs), 0) + b"".join(relocs) + bytes(slots))
        except _NotPlannable as e:
            self.failed = str(e)


class _Plan:
    def __init__(self, version, blob, scratch, keep):
        self.version, self.blob, self.scratch, self.keep = version, blob, scratch, keep

    def run(self, tensors):
        t0 = tensors[0]
        scratch = torch.empty(self.scratch, dtype=torch.uint8, device=t0.device) if self.scratch else None
        n = len(tensors) + 2
        bases = (ctypes.c_uint64 * n)(0, scratch.data_ptr() if self.scratch else 0,
                                      *[0 if t is None else t.data_ptr() for t in tensors])
        _lib.call("ffk_run_plan", self.blob, len(self.blob), bases, n, _lib.stream_ptr())


class _Watch:
    """The parameters of a module tree, found once and again whenever a sub-module has been exchanged."""

    def __init__(self, owner):
        mods = list(owner.modules())
        self.children = [(m._modules, list(m._modules.values())) for m in mods if m._modules]
        self.params = [m._parameters for m in mods if m._parameters]
        self.mods = mods

    def intact(self):
        return all(list(d.values()) == seen for d, seen in self.children)

    def version(self):
        return [epoch] + [(p.data_ptr(), p._version) for d in self.params for p in d.values() if p is not None]

    def tensors(self):
        """Parameters and everything the modules have packed from them."""
        out = [p for d in self.params for p in d.values() if p is not None]

        def walk(v):
            if isinstance(v, torch.Tensor):
                out.append(v)
                for extra in v.__dict__.values():       # e.g. a packing of a subset of the rows
                    walk(extra)
            elif isinstance(v, (tuple, list)):
                for x in v:
                    walk(x)
            elif hasattr(v, "buf"):
                walk(v.buf)
        for m in self.mods:
            for _, packed in m.__dict__.get("_pack_cache", {}).values():
                walk(packed)
        return out


class _State:
    """Per-module state of ``run``; not part of copies."""

    def __init__(self, owner):
        self.watch = _Watch(owner)
        self.plans = OrderedDict()               # the one used longest ago first
        self.lock = threading.Lock()             # of the order and the size of ``plans``

    def touch(self, key):
        with self.lock:
            if key in self.plans:                # another thread may have dropped it since
                self.plans.move_to_end(key)

    def store(self, key, plan):
        with self.lock:
            self.plans[key] = plan
            self.plans.move_to_end(key)
            while len(self.plans) > _MAX_PLANS:
                self.plans.popitem(last=False)

    def __deepcopy__(self, memo):
        return None

    def __reduce__(self):
        return type(None), ()


def alloc(t):
    """Reports a scratch tensor of the running sequence."""
    rec = _lib._STATE.recorder
    if rec is not None:
        rec.alloc(t)
    return t


def scope():
    rec = _lib._STATE.recorder
    if rec is not None:
        rec.scope()


def hold():
    rec = _lib._STATE.recorder
    if rec is not None:
        rec.hold()


def _sharing(tensors):
    """Which of the tensors share memory, and how: () or one (position, position of another, bytes between their starts) per
    tensor that begins inside memory another one has begun in.  A recording knows a buffer by its address only, so a plan fits
    no call in which other buffers coincide (one mask passed for both, a cotangent that is the input itself)."""
    spans = sorted((t.data_ptr(), i, t.nbytes) for i, t in enumerate(tensors) if t is not None)
    out, start, first, end = [], 0, 0, 0
    for lo, i, n in spans:
        if lo < end:
            out.append((i, first, lo - start))
        else:
            start, first = lo, i
        end = max(end, lo + n)
    return tuple(sorted(out))            # in the order of the list, whatever the addresses


def run(owner, key, tensors, sequence):
    """Executes ``sequence()`` - launches on the current stream that work on ``tensors`` (a list, entries may be None; the
    first is not), on scratch from ``alloc`` and on the weights of the module ``owner`` - or replays its plan.  ``key``
    names everything else the launches depend on (shapes, dtypes, switches) but which of ``tensors`` share memory."""
    if _lib._TIMED or _lib._STATE.recorder is not None:        # launches are being timed one by one, or recorded already
        return sequence()
    st = owner.__dict__.get("_plan_state")
    if st is None or not st.watch.intact():
        st = owner.__dict__["_plan_state"] = _State(owner)
    version = st.watch.version()
    key = (key, _sharing(tensors))
    plan = st.plans.get(key)
    if plan is not None and plan.version == version:
        st.touch(key)
        if plan.blob is None:
            return sequence()
        return plan.run(tensors)
    if any(p.dtype != tensors[0].dtype for d in st.watch.params for p in d.values() if p is not None):
        return sequence()        # parameters of another dtype are converted on the way, into memory no recording knows
    before = builds
    rec = _lib._STATE.recorder = _Recorder(tensors, st.watch.tensors())
    try:
        sequence()
    finally:
        _lib._STATE.recorder = None
    if builds != before:
        return           # weights were packed on the way: their memory was not known when the recording began
    st.store(key, _Plan(version, None if rec.failed else b"".join(rec.out), rec.peak, st.watch.tensors()))

"""What the optimizers' batches of steps hand to the library, by a library that records the
calls in place of launching kernels (host-only entry points are the real library's)."""
import ctypes
import struct

import pytest
import torch

from muon_sr_amd import _lib, adamw_8bit
from muon_sr_amd.adamw_8bit import _Adam8Batch, init_8bit_state
from muon_sr_amd.muon import _MuonEach

# item layouts and the place of the parameter's address
ITEM = {"msr_adamw8bit_multi": (struct.Struct("=QQQQQQqIi"), 0), "msr_adamw_multi": (struct.Struct("=QQQQqffIi"), 0),
        "msr_muon_each": (struct.Struct("=QQQqqIIif"), 2)}
OVERLAP = 1005


class Recorder:
    """Stands in for the library: ``calls`` holds (entry point, parameter addresses).  A list with
    an address in ``refuse`` is refused."""

    def __init__(self, real):
        self.real, self.calls, self.refuse = real, [], set()

    def msr_adamw8bit_apart(self, q, nq, block, b, nb, apart):
        for name, items in (("msr_adamw8bit_multi", q), ("msr_adamw_multi", b)):
            step, at = ITEM[name]
            if self.refuse & {x[at] for x in step.iter_unpack(items)}:
                apart._obj.value = 0
                return 0
        return self.real.msr_adamw8bit_apart(q, nq, block, b, nb, apart)

    def __getattr__(self, name):
        if name not in ITEM:
            return getattr(self.real, name)

        def call(items, count, *rest):
            step, at = ITEM[name]
            assert len(items) == count * step.size
            ps = [step.unpack_from(items, i * step.size)[at] for i in range(count)]
            if self.refuse & set(ps):
                return OVERLAP
            self.calls.append((name, ps))
            return 0
        return call


@pytest.fixture
def rec(monkeypatch):
    rec = Recorder(_lib.lib())
    monkeypatch.setattr(_lib, "lib", lambda: rec)
    monkeypatch.setattr(_lib, "stream_of", lambda t: 0)
    monkeypatch.setattr(adamw_8bit, "quant_table", lambda state: 64)
    return rec


@pytest.fixture
def calls(rec):
    return rec.calls


def _add8(batch, p, maps, numel8=4096):
    state = init_8bit_state(p, 256, 8, numel8, maps)
    state["step"] = 1
    grad = torch.zeros_like(p)
    batch.add(p, grad, state, 7)
    return state, grad   # kept by the caller until the flush, as an optimizer's are


def test_8bit_kinds_that_share_memory_run_in_order(calls):
    """A bf16-moment tensor that is a view of a quantized one: steps as added, whichever comes first."""
    maps, keep = {}, []
    flat = torch.zeros(20000, dtype=torch.bfloat16)
    small, whole = flat[100:300], flat[:8192]
    other = torch.zeros(9000, dtype=torch.bfloat16)
    for order in ([small, whole], [whole, small], [other, small, whole, flat[8192:8200]]):
        calls.clear()
        batch = _Adam8Batch(1e-3, 0.9, 0.99, 1e-8, 0.0)
        keep.append([_add8(batch, p, maps) for p in order])
        batch.flush()
        assert [a for _, items in calls for a in items] == [p.data_ptr() for p in order]


def test_8bit_kinds_that_share_nothing_take_two_launches(calls):
    """Neighbouring views of one buffer do not overlap: one launch of each kind."""
    maps, keep = {}, []
    flat = torch.zeros(40000, dtype=torch.bfloat16)
    views = flat.split([8192, 64, 8192, 64, 8192, 15296])
    batch = _Adam8Batch(1e-3, 0.9, 0.99, 1e-8, 0.0)
    keep += [_add8(batch, p, maps) for p in views]
    batch.flush()
    assert sorted((name, len(items)) for name, items in calls) == [("msr_adamw8bit_multi", 4), ("msr_adamw_multi", 2)]


def test_refused_item_ends_the_list(rec):
    """An item that the library refuses: the earlier ones are stepped, it and the later ones are not,
    and the later ones' steps are taken back, in every kind of batch."""
    maps = {}
    ps = [torch.zeros(n, dtype=torch.bfloat16) for n in (8192, 64, 8192, 64, 8192, 64)]
    for bad in range(len(ps)):
        rec.calls.clear()
        rec.refuse = {ps[bad].data_ptr()}
        batch = _Adam8Batch(1e-3, 0.9, 0.99, 1e-8, 0.0)
        kept = [_add8(batch, p, maps) for p in ps]
        with pytest.raises(_lib.MuonSRLibraryError):
            batch.flush()
        assert [a for _, items in rec.calls for a in items] == [p.data_ptr() for p in ps[:bad]]
        assert [s["step"] for s, _ in kept] == [1] * (bad + 1) + [0] * (len(ps) - bad - 1)


def test_refused_matrix_ends_the_list(rec):
    ps = [torch.zeros(64, 96, dtype=torch.bfloat16) for _ in range(5)]
    rec.refuse = {ps[3].data_ptr()}
    each = _MuonEach(0.95, True, 5, 0.02, 0.0)
    states = [dict(step=1, buf=torch.zeros_like(p)) for p in ps]
    for i, (p, s) in enumerate(zip(ps, states)):
        p.grad = torch.zeros_like(p)
        each.add(p, s["buf"], s["step"], i, s)
    with pytest.raises(_lib.MuonSRLibraryError):
        each.flush()
    assert [a for _, items in rec.calls for a in items] == [p.data_ptr() for p in ps[:3]]
    assert [s["step"] for s in states] == [1, 1, 1, 1, 0]


def test_matrices_one_by_one_where_memory_runs_out(rec, monkeypatch):
    """The list's workspace does not fit: one matrix at a time, each with its own smaller workspace."""
    real, sizes = torch.empty, []

    def empty(n, **kw):
        sizes.append(n)
        if len(sizes) == 1:
            raise torch.OutOfMemoryError("no memory for the list")
        return real(n, **kw)
    ps = [torch.zeros(64, 96, dtype=torch.bfloat16) for _ in range(4)]
    each = _MuonEach(0.95, True, 5, 0.02, 0.0)
    states = [dict(step=1, buf=torch.zeros_like(p)) for p in ps]
    for i, (p, s) in enumerate(zip(ps, states)):
        p.grad = torch.zeros_like(p)
        each.add(p, s["buf"], s["step"], i, s)
    monkeypatch.setattr(torch, "empty", empty)
    each.flush()
    assert [items for _, items in rec.calls] == [[p.data_ptr()] for p in ps]
    assert [s["step"] for s in states] == [1] * 4 and max(sizes[1:]) < sizes[0]


def test_apart_checks_the_items():
    """An item that the step would refuse (p and g overlap in part) is never apart; equal buffers and
    empty items are."""
    L, apart = _lib.lib(), ctypes.c_int32(-1)
    q8, b16 = ITEM["msr_adamw8bit_multi"][0].pack, ITEM["msr_adamw_multi"][0].pack
    q = q8(1 << 20, 2 << 20, 3 << 20, 4 << 20, 5 << 20, 6 << 20, 1000, 1, 0)
    for p, g, n, want in ((7 << 20, 8 << 20, 1000, 1), (7 << 20, (7 << 20) + 16, 1000, 0), (7 << 20, 7 << 20, 1000, 1),
                          ((1 << 20) + 1998, 8 << 20, 1000, 0), ((1 << 20) + 2000, 8 << 20, 1000, 1), (1 << 20, 8 << 20, 0, 1),
                          (7 << 20, 8 << 20, -1, 0), (0, 8 << 20, 1000, 0), (7 << 20, 2 << 20, 1000, 1)):
        b = b16(p, g, 9 << 20, 10 << 20, n, 0.1, 0.1, 1, 0)
        assert L.msr_adamw8bit_apart(q, 1, 256, b, 1, ctypes.byref(apart)) == 0
        assert apart.value == want, (p, g, n)
    assert L.msr_adamw8bit_apart(q, 1, 0, None, 0, ctypes.byref(apart)) == 1001


@pytest.mark.parametrize("which", ["8bit", "hybrid"])
def test_loaded_states_share_launches(rec, which):
    """After load_state_dict the quantized tensors take one launch, as a new optimizer's do: states whose
    codebooks have the same bits share one pair, beside parameters whose state begins later, and
    other codebooks keep theirs."""
    import copy
    from muon_sr_amd import TritonAdamW8bit, TritonMuonSRWithAuxAdam
    ps = [torch.nn.Parameter(torch.zeros(64, 96, dtype=torch.bfloat16)) for _ in range(6)]

    def make():
        if which == "8bit":
            return TritonAdamW8bit(ps, lr=1e-3)
        return TritonMuonSRWithAuxAdam([dict(params=ps, use_muon=False, optim_bits=8)])

    def launches(opt):
        rec.calls.clear()
        batch = _Adam8Batch(1e-3, 0.9, 0.99, 1e-8, 0.0)
        kept = []
        for p in ps:
            state = opt.state[p] or opt.state[p].update(init_8bit_state(p, 256, 8, 4096, opt._maps)) or opt.state[p]
            state["step"] = 3
            kept.append(torch.zeros_like(p))
            batch.add(p, kept[-1], state, 7)
        batch.flush()
        return [len(items) for _, items in rec.calls]

    opt = make()
    assert launches(opt) == [6]
    saved = copy.deepcopy(opt.state_dict())
    for st in saved["state"].values():   # a pair per state, as an earlier load made them
        st["qmap1"], st["qmap2"] = st["qmap1"].clone(), st["qmap2"].clone()
    del saved["state"][2]                # a parameter that had no gradient yet
    opt = make()
    opt.load_state_dict(saved)
    assert launches(opt) == [6]
    opt = copy.deepcopy(make())
    opt.load_state_dict(saved)
    saved["state"][4]["qmap1"][3] += 1e-3
    saved["state"][5]["qmap1"][3] += 1e-3
    opt = make()
    opt.load_state_dict(saved)
    assert launches(opt) == [4, 2]
    for i, st in saved["state"].items():
        for key in ("qmap1", "qmap2"):
            assert torch.equal(opt.state[ps[i]][key], st[key]) and opt.state[ps[i]][key].data_ptr() != st[key].data_ptr()

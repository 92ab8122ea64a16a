"""What the optimizers' batches of steps hand to the library, by a library that records the
calls in place of launching kernels (host-only entry points are the real library's)."""
import struct

import pytest
import torch

from muon_sr_amd import _lib, adamw_8bit
from muon_sr_amd.adamw_8bit import _Adam8Batch, init_8bit_state

ITEM = {"msr_adamw8bit_multi": struct.Struct("=QQQQQQqIi"), "msr_adamw_multi": struct.Struct("=QQQQqffIi")}


class Recorder:
    """Stands in for the library: ``calls`` holds (entry point, parameter addresses)."""

    def __init__(self, real):
        self.real, self.calls = real, []

    def __getattr__(self, name):
        if name not in ITEM:
            return getattr(self.real, name)

        def call(items, count, *rest):
            step = ITEM[name]
            assert len(items) == count * step.size
            self.calls.append((name, [step.unpack_from(items, i * step.size)[0] for i in range(count)]))
            return 0
        return call


@pytest.fixture
def calls(monkeypatch):
    rec = Recorder(_lib.lib())
    monkeypatch.setattr(_lib, "lib", lambda: rec)
    monkeypatch.setattr(_lib, "stream_of", lambda t: 0)
    monkeypatch.setattr(adamw_8bit, "quant_table", lambda state: 64)
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

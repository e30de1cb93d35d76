"""The code tables that quantize_4bit keeps per device: what a tracing or fake-tensor pass makes of them stays its own."""
from __future__ import annotations

import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode

from molt_amd import nf4


class _Mode(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_fake_and_traced_calls_leave_no_tables_behind(monkeypatch):
    monkeypatch.setattr(nf4, "_TABLES", {})
    dev = torch.device("cuda:0")
    with FakeTensorMode(allow_non_fake_inputs=True):
        fake = nf4._tables(dev)
        packed, qs = nf4.quantize_4bit(torch.empty(64, 64, device=dev, dtype=torch.bfloat16))
    assert type(fake[0]).__name__ == type(packed).__name__ == type(qs.code).__name__ == "FakeTensor"
    assert nf4._TABLES == {}
    cpu = torch.device("cpu", 0)
    with _Mode():
        nf4._tables(cpu)
    torch.func.vmap(lambda x: x + nf4._tables(cpu)[0].sum())(torch.zeros(2))
    assert nf4._TABLES == {}
    with torch.inference_mode():
        kept = nf4._tables(cpu)
    assert nf4._tables(cpu) is kept and [type(t) for t in kept] == [torch.Tensor] * 2
    assert not any(t.is_inference() for t in kept) and torch.equal(kept[1], nf4.dynamic_map())

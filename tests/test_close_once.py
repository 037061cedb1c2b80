"""A handle is destroyed once, also when its owner is collected while the interpreter shuts down and the modules'
names are gone already."""
import ctypes

import pytest

from mithra_amd import abi, job


class Library:
    """Counts the destructions of each handle."""

    def __init__(self):
        self.destroyed = []

    def __getattr__(self, name):
        return lambda h: self.destroyed.append(h) or 0


@pytest.mark.parametrize("module,kind", [(abi, "Domain"), (abi, "DeviceBunch"), (abi, "Batch"), (abi, "MLP"),
                                         (job, "Job")])
def test_destroyed_once(module, kind, monkeypatch):
    cls = getattr(module, kind)
    owner = cls.__new__(cls)
    owner.lib = Library()
    owner.f = {"destroy": owner.lib.destroy}
    owner.h = ctypes.c_void_p(1234)
    monkeypatch.setattr(module, "C", None)
    for _ in range(3):
        owner.__del__()
    owner.close()
    assert len(owner.lib.destroyed) == 1

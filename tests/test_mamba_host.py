"""CPU: which of a block's row functions mamba.mamba_verify runs."""
import types

import pytest
import torch

from hsd import mamba
from hsd import model as Mdl


class Scaled(Mdl.MambaBlock):
    def rows(self, x, buf, cache, status=None):
        return x.mul_(3)


class Proxy:
    """Another block's attributes, and rows of its own."""

    def __init__(self, inner):
        self.inner = inner

    def __getattr__(self, name):
        return getattr(self.inner, name)

    def rows(self, x, buf, cache, status=None):
        return x.mul_(3)


def stub(cls):
    b = cls.__new__(cls)
    b.in_proj, b.norm_w = types.SimpleNamespace(O=32), torch.ones(16)
    b.mixer = types.SimpleNamespace(intermediate_size=16)
    return b


def patched():
    b = stub(Mdl.MambaBlock)
    b.rows = lambda x, buf, cache, status=None: x.mul_(3)
    return b


@pytest.mark.parametrize("make", [lambda: stub(Scaled), lambda: Proxy(stub(Mdl.MambaBlock)), patched])
def test_a_block_with_its_own_rows(make, monkeypatch):
    monkeypatch.setattr(Mdl.MambaBlock, "rows_into", lambda self, x, buf, cache, out, status=None: out.copy_(x))
    x, records = torch.arange(48.0).view(1, 3, 16).to(torch.bfloat16), []
    y = mamba.mamba_verify(make(), x, "cache", records)
    assert torch.equal(y, 3 * x) and records == [("cache", 3)] and float(x[0, 0, 1]) == 1.0
    z = mamba.mamba_verify(stub(Mdl.MambaBlock), x, "cache", records)      # its own class: out of place
    assert torch.equal(z, x) and z.data_ptr() != x.data_ptr()

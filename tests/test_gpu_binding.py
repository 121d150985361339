"""GPU: the native binding's pointer arguments."""
import pytest
import torch

from hsd import _native as N

pytestmark = pytest.mark.gpu


def test_copy_on_write(dev):
    """A lazy clone that an entry point writes gets memory of its own; one that it only reads
    does not need to."""
    a = torch.arange(16, dtype=torch.int32, device=dev)
    b = torch._lazy_clone(a)
    N.call("hsd_seq_add", b, 3, 5, N.stream(dev))
    assert a.tolist() == list(range(16)) and b.tolist() == [0, 1, 2, 8] + list(range(4, 16))
    src, dst = torch._lazy_clone(a), torch.zeros(2, dtype=torch.int32, device=dev)
    seq = torch.zeros(16, dtype=torch.int32, device=dev)
    N.call("hsd_prompt_tokens", src, 16, seq, 1, 2, dst, N.stream(dev))
    assert dst.tolist() == [1, 2]

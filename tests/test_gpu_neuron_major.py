"""GPU: layout.to_neuron_major in one launch against its three separate permutations, bit for
bit, at the edges of its 32-word tiles and 128-row pieces, and past its 64 groups."""
import pytest
import torch

from hsd import layout

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lead,R,G", [((), 8, 1), ((3,), 120, 2), ((2,), 128, 29), ((2,), 136, 64), ((), 264, 65), ((2, 2), 72, 3)])
def test_one_launch_equals_three(dev, lead, R, G):
    g = torch.Generator(device=dev)
    g.manual_seed(R + G)
    w = torch.randint(-2 ** 31, 2 ** 31, (*lead, R, 8 * G), dtype=torch.int32, device=dev, generator=g)
    s, b = (torch.randint(-2 ** 15, 2 ** 15, (*lead, R, G), dtype=torch.int16, device=dev, generator=g) for _ in range(2))
    got = layout.to_neuron_major(w, s, b)
    want = layout.nibble_transpose(w), layout.transpose_last2(s), layout.transpose_last2(b)
    for x, y in zip(got, want):
        assert x.shape == y.shape and x.dtype == y.dtype and torch.equal(x, y)
    # scales that are not 16-byte aligned take the separate launches
    so = torch.empty(s.numel() + 1, dtype=s.dtype, device=dev)[1:].view(s.shape).copy_(s)
    assert torch.equal(layout.to_neuron_major(w, so, b)[1], want[1])

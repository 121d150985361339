"""CPU: which launches layout.to_neuron_major makes (shapes only: no tensor here has memory)."""
import pytest
import torch

from hsd import _native as N
from hsd import layout


@pytest.mark.parametrize("R,G,one", [(128, 29, True), (2 ** 25 - 8, 64, True), (2 ** 25, 64, False), (64, 65, False),
                                     (64, 0, False)])
def test_one_launch_or_three(monkeypatch, R, G, one):
    """Scales of more than 2^31 - 1 values per matrix go through the separate permutations."""
    calls = []
    monkeypatch.setattr(N, "call", lambda name, *a: calls.append(name))
    monkeypatch.setattr(N, "stream", lambda device=None: 0)
    w = torch.empty((R, 1), dtype=torch.int32, device="meta")
    s, b = (torch.empty((R, G), dtype=torch.bfloat16, device="meta") for _ in range(2))
    got = layout.to_neuron_major(w, s, b)
    assert [t.shape for t in got] == [(8, R // 8), (G, R), (G, R)]
    assert calls == (["hsd_neuron_major"] if one else ["hsd_permute_nibbles", "hsd_transpose_u16", "hsd_transpose_u16"])

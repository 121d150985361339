"""The sparse down projection with two weight words per lane (many token rows): an output's
sums run over the same values in the same order as with one word, so every row of a call
equals the same row in a call of its own, bit for bit, at the rule's edges: the row counts on
both sides of it, a last chunk of 128 of its 256 outputs, weights that two words' loads
cannot take, and each activation type."""
import pytest
import torch

from hsd import decode

pytestmark = pytest.mark.gpu
F, FS, TOPK, E = 128, 192, 3, 5


@pytest.mark.parametrize("B", [3, 4, 9])
@pytest.mark.parametrize("D", [128, 256, 384, 640])
@pytest.mark.parametrize("off", [0, 1])
def test_rows_equal_single_rows(dev, B, D, off):
    gen = torch.Generator().manual_seed(B * D + off)

    def words(*shape):
        n = torch.Size(shape).numel()
        w = torch.randint(-2 ** 31, 2 ** 31, (n + off,), generator=gen, dtype=torch.int64).to(torch.int32).to(dev)
        return w[off:].view(shape)

    def bf(*shape):
        return torch.randn(shape, generator=gen).to(torch.bfloat16).to(dev)

    nm = (words(E, F, D // 8), bf(E, F // 64, D), bf(E, F // 64, D), words(FS, D // 8), bf(FS // 64, D), bf(FS // 64, D))
    h = torch.randn((B, TOPK * F + FS), generator=gen) * (torch.rand((B, TOPK * F + FS), generator=gen) < 0.3)
    h[-1] = 0.0                                       # a row with nothing live
    sel = torch.randint(0, E, (B, TOPK), generator=gen, dtype=torch.int32).to(dev)
    gains = torch.rand((B, TOPK + 1), generator=gen).to(dev)
    kw = dict(F=F, FS=FS, D=D, topk=TOPK, out_dtype=torch.float32)
    for dt in (torch.bfloat16, torch.float16, torch.float32):
        hd = h.to(dt).to(dev)
        y = decode.sparse_down(hd, sel, gains, *nm, **kw)
        assert torch.equal(y, decode.sparse_down(hd, sel, gains, *nm, dense=True, **kw))
        assert not y[-1].any()
        for b in range(B):
            assert torch.equal(y[b:b + 1], decode.sparse_down(hd[b:b + 1], sel[b:b + 1], gains[b:b + 1], *nm, **kw))

"""GPU: MoEBlock.prefill_sparse on both sides of its rule. Up to CHUNK_MIN rows its bits are those
of the front end and the down projection over each tile's union of live rows; above, the two
paths differ by fp32 summation orders: a bf16 rounding of h (2^-9 relative, squared) in some of
a row's neurons and one of the projection, far below 2^-6 of the update."""
import pytest
import torch

from hsd import model as Mdl
from hsd import prefill as P

pytestmark = pytest.mark.gpu
CFG = Mdl.ModelConfig(hidden=512, n_experts=16, topk=3, moe_inter=256, shared_inter=512)


def block(dev):
    return Mdl.MoEBlock(CFG, Mdl._Init(3, dev))


def rows(dev, T):
    g = torch.Generator(device=dev)
    g.manual_seed(T)
    return torch.randn((T, CFG.hidden), device=dev, generator=g).to(torch.bfloat16)


def by_union(blk, x, tt):
    h, sel, gains = blk._front_packed(x)
    tiles = P.build_tiles(sel, CFG.n_experts, tt)
    kw = dict(F=CFG.moe_inter, FS=CFG.shared_inter, topk=CFG.topk, E=CFG.n_experts, tt=tt)
    union = P.build_union(h, *tiles, **kw)
    y = P.sparse_down_prefill(h, sel, gains, blk.pw, blk.ps, blk.pb, blk.spw, blk.sps, blk.spb, D=CFG.hidden,
                              tiles=tiles, union=union, **kw)
    return x + y.to(x.dtype)


@pytest.mark.parametrize("tt", [32, 64])
@pytest.mark.parametrize("T", [1, 4, 5, 12, 13, 40])
def test_rule(dev, T, tt):
    blk, x = block(dev), rows(dev, T)
    y, ref = blk.prefill_sparse(x, tt), by_union(blk, x, tt)
    if T <= 12:
        assert torch.equal(y.view(torch.int16), ref.view(torch.int16))
    else:
        assert float((y.double() - ref.double()).norm()) <= 2.0 ** -6 * float((ref.double() - x.double()).norm())


@pytest.mark.parametrize("T", [12, 13])
def test_leaves_no_statistics(dev, T):
    """The zero fractions of a layer's `trace` are those of the model's own rows: a call of the
    block by itself adds none (and reads nothing back to the host)."""
    blk = block(dev)
    blk.trace = []
    blk.prefill_sparse(rows(dev, T))
    assert blk.trace == []
    blk.chunk(rows(dev, T))
    assert len(blk.trace) == 1


WEIGHTS = ("w1", "s1", "b1", "sw1", "ss1", "sb1", "pw", "ps", "pb", "spw", "sps", "spb")


@pytest.mark.parametrize("T", [12, 40])
def test_strided_weights(dev, T):
    """Weights that are views of wider tensors (a checkpoint's fused ones) count like their
    contiguous copies."""
    blk, x = block(dev), rows(dev, T)
    want = blk.prefill_sparse(x)
    for n in WEIGHTS:
        t = getattr(blk, n)
        wide = torch.zeros((*t.shape[:-1], 2 * t.shape[-1]), dtype=t.dtype, device=dev)
        wide[..., :t.shape[-1]] = t
        setattr(blk, n, wide[..., :t.shape[-1]])
        assert not getattr(blk, n).is_contiguous()
        assert torch.equal(blk.prefill_sparse(x).view(torch.int16), want.view(torch.int16)), n


@pytest.mark.parametrize("name", ["pw", "spw"])
def test_words_at_any_address(dev, name):
    """Down weights at a multiple of 4 bytes only, which the chunk's 16-byte loads do not take,
    go through the union lists."""
    blk, x = block(dev), rows(dev, 40)
    assert blk.chunkable()
    t = getattr(blk, name)
    setattr(blk, name, torch.zeros(t.numel() + 1, dtype=t.dtype, device=dev)[1:].view(t.shape).copy_(t))
    assert not blk.chunkable()
    assert torch.equal(blk.prefill_sparse(x).view(torch.int16), by_union(blk, x, 32).view(torch.int16))

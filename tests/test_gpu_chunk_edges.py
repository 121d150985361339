"""GPU: the prompt-chunk products past the edges of their dispatch: the 64-row ring kernel and the
ring kernel at 4096 inputs (the projections of a long prompt), weights that only the ring kernel
takes, ids of no expert, rows that are not finite, and a call cut into several. Bounds as in
test_gpu_chunk: exact products, fp32 sums, one bf16 rounding (2^-9) of each result."""
import numpy as np
import pytest
import torch

from hsd import _native as N
from hsd import chunk, layout, nn
from hsd import model as Mdl
from tests.test_gpu_chunk import close, deq, rand

pytestmark = pytest.mark.gpu


def shifted(t, n=2):
    """t at an address of 4 bytes past a multiple of 16."""
    return torch.zeros(t.numel() + n, dtype=t.dtype, device=t.device)[n:].view(t.shape).copy_(t)


def bits(t):
    return t.contiguous().view(torch.int16)


# (64-row ring: 11 output blocks x 25 row tiles >= 256; 4096 inputs past 256 rows: the ring, with
# 32 rows and with 64)
@pytest.mark.parametrize("T,O,I", [(1537, 2696, 640), (257, 104, 4096), (1537, 2696, 4096), (1600, 2688, 128)])
def test_many_rows(dev, T, O, I):
    W = nn.QWeight(*Mdl._Init(T + O, dev).q4(O, I, 1.0 / np.sqrt(I)))
    x = rand(dev, T, T, I).to(torch.bfloat16)
    rows, ref = chunk.prep(x), x.double() @ deq(W.w, W.scales, W.biases).t().contiguous()
    assert close(chunk.gemm(rows, W), ref)
    res = rand(dev, 7, T, O).to(torch.bfloat16)
    y = chunk.gemm(rows, W, residual=res)
    assert close(y, res.double() + ref, inner=ref)
    z = res.clone()
    assert torch.equal(bits(chunk.gemm(rows, W, residual=z, out=z)), bits(y))


@pytest.mark.parametrize("T", [5, 64, 256])
@pytest.mark.parametrize("O", [32, 40, 72, 104])
def test_in_place_residual_of_4096_inputs(dev, T, O):
    """The last 32 outputs of O end at O and overlap the ones before: each is written once."""
    W = nn.QWeight(*Mdl._Init(O, dev).q4(O, 4096, 1.0 / 64))
    rows, res = chunk.prep(rand(dev, T, T, 4096).to(torch.bfloat16)), rand(dev, 7, T, O).to(torch.bfloat16)
    z = res.clone()
    assert torch.equal(bits(chunk.gemm(rows, W, residual=z, out=z)), bits(chunk.gemm(rows, W, residual=res)))


@pytest.mark.parametrize("T,O,I", [(33, 328, 640), (64, 72, 4096), (5, 64, 128)])
def test_scales_at_four_bytes(dev, T, O, I):
    """Scales that the 16-byte loads of the register kernels do not take: the ring kernel."""
    w, s, b = Mdl._Init(O, dev).q4(O, I, 1.0 / np.sqrt(I))
    x = rand(dev, T, T, I).to(torch.bfloat16)
    y = chunk.gemm(chunk.prep(x), nn.QWeight(w, shifted(s), shifted(b)))
    assert close(y, x.double() @ deq(w, s, b).t().contiguous())


E, D, F, FS, K = 16, 256, 192, 320, 3


def layer(dev, seed):
    init = Mdl._Init(seed, dev)
    up = [*init.q4(F, D, 1.0 / np.sqrt(D), lead=(E,)), *init.q4(FS, D, 1.0 / np.sqrt(D))]
    down = [*layout.to_neuron_major(*init.q4(D, F, 1.0 / np.sqrt(F), lead=(E,))),
            *layout.to_neuron_major(*init.q4(D, FS, 1.0 / np.sqrt(FS)))]
    return up, down


def run(x, sel, gains, up, down, tt, status=None):
    rows, tiles = chunk.prep(x), chunk.moe_tiles(sel, E, tt, status=status)
    h, hsum = chunk.moe_up(rows, tiles, *up, topk=K, tt=tt)
    return chunk.moe_down(x, h, hsum, sel, gains, tiles, *down, topk=K, tt=tt), h


def routing(dev, T, seed):
    rng = np.random.default_rng(seed)
    sel = torch.from_numpy(np.stack([rng.permutation(E)[:K] for _ in range(T)]).astype(np.int32)).to(dev)
    return sel, rand(dev, seed + 1, T, K + 1).abs()


def test_up_scales_at_four_bytes(dev):
    """The expert products' ring kernel with 32-slot tiles against the register kernel: two fp32
    sums of u may round to neighbouring bf16 values, whose squares differ by 2^-6 and a rounding."""
    up, _ = layer(dev, 3)
    x = rand(dev, 1, 70, D).to(torch.bfloat16)
    sel, _ = routing(dev, 70, 5)
    rows, tiles = chunk.prep(x), chunk.moe_tiles(sel, E, 32)
    odd = [shifted(t) if i % 3 else t for i, t in enumerate(up)]
    (h, s), (g, u) = (chunk.moe_up(rows, tiles, *w, topk=K, tt=32) for w in (up, odd))
    h, g = h.double(), g.double()
    assert bool(((h - g).abs() <= (2.0 ** -6 + 2.0 ** -7) * h + 1e-4 * h.max()).all())
    n = [slice(0, F // 64)] * K + [slice(0, FS // 64)]
    gp = s.shape[2] // 3
    for k in range(K + 1):
        a, b = (sum(t[:, k, i * gp:(i + 1) * gp][:, n[k]].double() for i in range(3)) for t in (s, u))
        assert bool(((a - b).abs() <= 2.0 ** -6 * a + 1e-3 * a.max()).all()), k


@pytest.mark.parametrize("T,tt", [(1, 32), (40, 32), (40, 64), (150, 64)])
def test_ids_of_no_expert(dev, T, tt):
    """Slots whose id is -1, E or far out add nothing, their h is not written, and the other
    slots' rows are those of a call where these go to an expert with gain zero."""
    up, down = layer(dev, 3)
    x = rand(dev, T, T, D).to(torch.bfloat16)
    sel, gains = routing(dev, T, 5)
    bad = sel.clone()
    hole = torch.rand((T, K), generator=torch.Generator().manual_seed(T)).to(dev) < 0.4
    hole[0, 0] = True
    bad[hole] = torch.tensor([-1, E, 1 << 30], dtype=torch.int32, device=dev).repeat(T * K)[:int(hole.sum())]
    status = torch.zeros(1, dtype=torch.int32, device=dev)
    y, _ = run(x, bad, gains, up, down, tt, status)
    assert int(status.item()) == N.STATUS_BAD_EXPERT
    zero = gains.clone()
    zero[:, :K][hole] = 0.0
    want, _ = run(x, sel, zero, up, down, tt)
    assert torch.equal(y, want)


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("T,tt", [(40, 32), (150, 64)])
def test_rows_that_are_not_finite(dev, T, tt, value):
    """Such a row spoils itself alone: the other rows of its tiles keep their bits, in the
    products of a layer, of a projection (register kernels, ring) and of a bf16 weight."""
    up, down = layer(dev, 3)
    x = rand(dev, T, T, D).to(torch.bfloat16)
    odd, r = x.clone(), T // 2
    odd[r, 17] = value
    keep = torch.arange(T, device=dev) != r
    sel, gains = routing(dev, T, 5)
    (a, ha), (b, hb) = (run(t, sel, gains, up, down, tt) for t in (x, odd))
    assert torch.equal(bits(a[keep]), bits(b[keep])) and torch.equal(bits(ha[keep]), bits(hb[keep]))
    assert not bool(torch.isfinite(b[r].float()).any())
    for O, I in ((328, D), (104, 4096)):
        w, s, bb = Mdl._Init(O, dev).q4(O, I, 1.0 / np.sqrt(I))
        dense = nn.QWeight(rand(dev, 9, O, I).to(torch.bfloat16))
        x = rand(dev, T, T, I).to(torch.bfloat16)
        odd = x.clone()
        odd[r, 17] = value
        nw = torch.ones(I, dtype=torch.bfloat16, device=dev)
        for W in (nn.QWeight(w, s, bb), nn.QWeight(w, shifted(s), shifted(bb)), dense):
            for norm in (None, nw):
                p, q = (chunk.gemm(chunk.prep(t, norm=norm), W) for t in (x, odd))
                assert torch.equal(bits(p[keep]), bits(q[keep]))
                assert not bool(torch.isfinite(q[r].float()).any())


@pytest.mark.parametrize("most", [1, 7, 32])
def test_a_call_cut_into_several(dev, most, monkeypatch):
    """More rows than one call's buffers take: the same rows in pieces, bit for bit (a row's sums
    do not depend on the rows beside it)."""
    cfg = Mdl.ModelConfig(hidden=512, n_experts=16, topk=3, moe_inter=256, shared_inter=512)
    blk = Mdl.MoEBlock(cfg, Mdl._Init(3, dev))
    x = rand(dev, 1, 45, 512).to(torch.bfloat16)
    want, z = blk.prefill_sparse(x), x.clone()
    monkeypatch.setattr(chunk, "moe_rows", lambda *a: most)
    assert torch.equal(bits(blk.prefill_sparse(x)), bits(want))
    assert torch.equal(bits(blk._chunk(z, 32, out=z)), bits(want))

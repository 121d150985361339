"""GPU: the prompt-chunk projections (hsd.chunk) against plain float64 torch on the same
weights, at the edges of their tiles: rows around the 32- and 64-row tiles, outputs that are
no multiple of 256, empty and crowded experts.

Bound: the kernels sum exact products (bf16 x 4-bit integers) in fp32 and round the result to
bf16 once, so an output is within half a bf16 ulp (2^-9 of its size) of the exact value plus
the fp32 sums' error, which is far below 1e-4 of the output's scale at these sizes."""
import numpy as np
import pytest
import torch

from hsd import chunk, layout, nn, prefill
from hsd import model as Mdl
from hsd.moe import up_relu2

pytestmark = pytest.mark.gpu


def deq(w, s, b):
    sh = torch.arange(0, 32, 4, device=w.device, dtype=torch.int32)
    q = ((w.unsqueeze(-1) >> sh) & 15).reshape(*w.shape[:-1], w.shape[-1] * 8).double()
    return q * s.double().repeat_interleave(64, -1) + b.double().repeat_interleave(64, -1)


def close(got, ref, inner=0.0):
    """inner: the exact product where it is rounded to bf16 once more before a residual add."""
    got, ref = got.double(), ref.double()
    scale = ref.abs().max()
    return bool(((got - ref).abs() <= 2.0 ** -8 * (ref.abs() + abs(inner)) + 2e-4 * scale).all())


def rand(dev, seed, *shape):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    return torch.randn(shape, device=dev, generator=g)


@pytest.mark.parametrize("T", [1, 31, 33, 64, 65, 200])
@pytest.mark.parametrize("O,I", [(64, 128), (328, 640), (2688, 512), (104, 2688), (72, 4096)])
def test_gemm_q4(dev, T, O, I):
    W = nn.QWeight(*Mdl._Init(T + O, dev).q4(O, I, 1.0 / np.sqrt(I)))
    x = rand(dev, T, T, I).to(torch.bfloat16)
    nw = (rand(dev, 5, I).abs() + 0.5).to(torch.bfloat16)
    rows = chunk.prep(x, norm=nw)
    ref_x = nn.linear(x, nn.QWeight(torch.zeros((4, I), dtype=torch.bfloat16, device=dev)), norm=nw,
                      xn_out=(xn := torch.empty_like(x)))
    del ref_x
    perm = torch.tensor([0, 4, 1, 5, 2, 6, 3, 7], device=dev)
    assert torch.equal(rows.xp.view(T, I // 8, 8), xn.view(T, I // 8, 8)[:, :, perm])
    ref = xn.double() @ deq(W.w, W.scales, W.biases).t().contiguous()
    assert close(chunk.gemm(rows, W), ref)
    res = rand(dev, 7, T, O).to(torch.bfloat16)
    y = chunk.gemm(rows, W, residual=res)
    assert close(y, res.double() + ref, inner=ref)
    # the bf16 weight on the same rows (permuted) and on natural ones
    wb = rand(dev, 9, O // 4 * 4, I).to(torch.bfloat16) / np.sqrt(I)
    Wb = nn.QWeight(wb)
    refb = xn.double() @ wb.double().t().contiguous()
    assert close(chunk.gemm(rows, Wb), refb)
    assert close(chunk.gemm(chunk.prep(x, norm=nw, sums=False), Wb), refb)


@pytest.mark.parametrize("T", [1, 33, 129, 400])
@pytest.mark.parametrize("O,I,sums", [(40, 24, False), (128, 640, True), (1312, 192, True), (1312, 192, False),
                                      (4100, 64, False)])
def test_gemm_bf16(dev, T, O, I, sums):
    """Both bf16 kernels (few and many tiles, the last one of each side cut), rows in either order."""
    W = nn.QWeight(rand(dev, O, O, I).to(torch.bfloat16))
    x = rand(dev, T, T, I).to(torch.bfloat16)
    y = chunk.gemm(chunk.prep(x, sums=sums), W).double()
    ref = x.double() @ W.w.double().t()
    assert bool(((y - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-4 * ref.abs().max()).all())


@pytest.mark.parametrize("T,tt", [(1, 32), (5, 32), (33, 64), (150, 32), (150, 64), (700, 64)])
def test_moe_up(dev, T, tt):
    E, D, F, FS, K = 16, 256, 192, 320, 3
    init = Mdl._Init(T, dev)
    w1, s1, b1 = init.q4(F, D, 1.0 / np.sqrt(D), lead=(E,))
    sw1, ss1, sb1 = init.q4(FS, D, 1.0 / np.sqrt(D))
    x = rand(dev, T, T, D).to(torch.bfloat16)
    rng = np.random.default_rng(T)
    # expert 0 in every row (crowded), experts 9..15 in none
    sel = np.stack([np.concatenate([[0], 1 + rng.permutation(8)[:K - 1]]) for _ in range(T)]).astype(np.int32)
    sel = torch.from_numpy(sel).to(dev)
    tiles = chunk.moe_tiles(sel, E, tt)
    te, ts = prefill.build_tiles(sel, E, tt)
    assert torch.equal(tiles[0], te) and torch.equal(tiles[1], ts)
    assert int(tiles[2].item()) == int((te[:T * K // tt + E] >= 0).sum().item())
    rows = chunk.prep(x)
    got, hsum = chunk.moe_up(rows, tiles, w1, s1, b1, sw1, ss1, sb1, topk=K, tt=tt)
    ref = up_relu2(x, sel, w1, s1, b1, sw1, ss1, sb1, topk=K)
    # square(relu(bf16(u))): two fp32 sums of u may round to neighbouring bf16 values (up to
    # 2^-7 apart, relative), whose squares differ by 2^-6 and round to bf16 (2^-9 each)
    g, r = got.double(), ref.double()
    bad = (g - r).abs() > (2.0 ** -6 + 2.0 ** -7) * r.abs() + 1e-4 * r.max()
    assert not bool(bad.any()), (g[bad][:8], r[bad][:8])
    assert float((g != r).double().mean()) < 0.02
    # the group sums: three bf16 parts hold the fp32 sum (64 values, within 2^-18 of exact)
    gp = hsum.shape[2] // 3
    hs = sum(torch.cat([hsum[:, :K, k * gp:k * gp + F // 64].reshape(T, -1), hsum[:, K, k * gp:k * gp + FS // 64]], 1).double()
             for k in range(3))
    want = g.view(T, -1, 64).sum(-1)
    assert bool(((hs - want).abs() <= 2.0 ** -18 * want.abs()).all())


@pytest.mark.parametrize("T,tt", [(1, 32), (5, 32), (33, 64), (150, 32), (150, 64), (700, 64)])
@pytest.mark.parametrize("D,F,FS,K", [(128, 64, 128, 6), (640, 192, 576, 3)])
def test_moe_down(dev, T, tt, D, F, FS, K):
    """Against the float64 sum over the layer's rows: fp32 sums of exact products, one bf16
    rounding of the projection and one of the residual sum (2^-9 each)."""
    E = 16
    init = Mdl._Init(T + D, dev)
    lay = [layout.to_neuron_major(*init.q4(D, F, 1.0 / np.sqrt(F), lead=(E,))),
           layout.to_neuron_major(*init.q4(D, FS, 1.0 / np.sqrt(FS)))]
    x = rand(dev, T, T, D).to(torch.bfloat16)
    h = torch.relu(rand(dev, T + 1, T, K * F + FS)).square().to(torch.bfloat16)
    h[:, 5:40] = 0
    gains = rand(dev, T + 2, T, K + 1).abs()
    rng = np.random.default_rng(T)
    sel = torch.from_numpy(np.stack([rng.permutation(9)[:K] for _ in range(T)]).astype(np.int32)).to(dev)
    gp = chunk.group_pitch(max(F, FS))
    hsum = torch.full((T, K + 1, 3 * gp), float("nan"), dtype=torch.bfloat16, device=dev)
    for k in range(K + 1):
        blk = h[:, k * F:(k + 1) * F] if k < K else h[:, K * F:]
        s = blk.float().view(T, -1, 64).sum(-1)
        n = s.shape[1]
        for i in range(3):
            hsum[:, k, i * gp:i * gp + n] = s.to(torch.bfloat16)
            s = s - hsum[:, k, i * gp:i * gp + n].float()
    tiles = chunk.moe_tiles(sel, E, tt)
    y = chunk.moe_down(x, h, hsum, sel, gains, tiles, *lay[0], *lay[1], topk=K, tt=tt)
    sh = torch.arange(0, 32, 4, device=dev, dtype=torch.int32)

    def rows(pw, ps, pb):
        q = ((pw.unsqueeze(-1) >> sh) & 15).reshape(*pw.shape[:-1], D).double()
        return q * ps.double().repeat_interleave(64, -2) + pb.double().repeat_interleave(64, -2)
    W, SW = rows(*lay[0]), rows(*lay[1])
    ref = gains[:, K:].double() * (h[:, K * F:].double() @ SW)
    for k in range(K):
        hk = h[:, k * F:(k + 1) * F].double()
        for e in range(9):
            m = sel[:, k] == e
            if bool(m.any()):
                ref[m] += gains[m, k:k + 1].double() * (hk[m] @ W[e])
    assert close(y, x.double() + ref, inner=ref)
    # in place over the residual
    z = x.clone()
    chunk.moe_down(z, h, hsum, sel, gains, tiles, *lay[0], *lay[1], topk=K, tt=tt, out=z)
    assert torch.equal(z.view(torch.int16), y.view(torch.int16))

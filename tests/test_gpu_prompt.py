"""GPU: the mixers of a prompt chunk (hsd.chunk.scan, hsd.chunk.attention) and the chunked
prompt against the decode kernels' row-by-row runs.

* scan: the state and the conv window bit-identical to mamba.ssm_rows in steps of up to 3 rows
  (the same arithmetic per element); z, whose sum over the 128 state elements has another
  order, within 2^-24 of the terms' sizes per addition (7 + 7 levels against 8 + 4: 2^-20 of
  sum |S C| covers both), and the 16-channel sums of z^2 accordingly;
* attention: the cache rows bit-exact, the outputs against float64 attention. The kernel sums
  exact bf16 products in fp32 and rounds once to bf16: half a bf16 ulp (2^-9) plus 2^-16 of
  the values' scale, doubled for the fp32 exponentials;
* prefill: both modes equal bits, and the caches near a run in 3-row steps. Two correct runs
  differ by bf16 roundings (a few 1e-3 after these layers) and, where a token's sixth and
  seventh experts are nearly tied, by one of six gains of that block's update of that row:
  with updates of at most the residual's size, sqrt(2)/6 of a row, which over T >= 4 rows
  and the blocks after it stays below 0.12/sqrt(T) + 2e-2 for one such token in four."""
import math

import numpy as np
import pytest
import torch

from hsd import _native as N
from hsd import chunk, mamba as M, nn
from hsd import model as Mdl

pytestmark = pytest.mark.gpu


def gen(dev, seed):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    return g


def mixer_and_state(dev, seed):
    blk = Mdl.MambaBlock(Mdl.ModelConfig(hidden=512, mtp=False), Mdl._Init(seed, dev))
    g = gen(dev, seed)
    m = blk.mixer
    conv = torch.randn((3, m.conv_dim), device=dev, generator=g).to(torch.bfloat16)
    ssm = torch.randn((m.num_heads, m.head_dim, m.ssm_state_size), device=dev, generator=g) * 0.1
    return m, conv, ssm, g


@pytest.mark.parametrize("T,cur0,pos0,total", [(1, 0, 0, 1), (2, 3, 0, 2), (15, 1, 0, 15), (16, 0, 0, 16), (17, 2, 0, 17),
                                               (33, 0, 5, 30), (40, 1, 9, 9)])
def test_scan_equals_rows(dev, T, cur0, pos0, total):
    m, conv, ssm, g = mixer_and_state(dev, T)
    width = 2 * m.intermediate_size + 2 * m.n_groups * m.ssm_state_size + m.num_heads
    proj = torch.randn((T, width), device=dev, generator=g).to(torch.bfloat16)
    cur = torch.full((1,), cur0, dtype=torch.int32, device=dev)
    pos = torch.full((1,), pos0, dtype=torch.int32, device=dev)
    ca = M.MambaCache(m, dev, nslab=4, cur=cur, conv_state=conv, ssm_state=ssm)
    cb = M.MambaCache(m, dev, nslab=4, cur=cur.clone(), conv_state=conv, ssm_state=ssm)
    z = chunk.scan(m, proj, ca, pos, total)
    V = min(max(total - pos0, 0), T)
    DI = m.intermediate_size
    for r in range(0, V, 3):
        n = min(3, V - r)
        zr = M.ssm_rows(m, proj[r:r + n], cb, gated=True)
        full = torch.as_strided(zr, (n, DI + DI // 16), (DI + DI // 16, 1))
        got = torch.as_strided(z, (T, DI + DI // 16), (DI + DI // 16, 1))[r:r + n]
        scale = full[:, :DI].abs().amax()        # sum |S C| is at most 16 times the largest |z| here
        assert float((got - full)[:, :DI].abs().max()) <= 2.0 ** -16 * float(scale), r
        assert float(((got - full)[:, DI:] / full[:, DI:]).abs().max()) <= 2.0 ** -12, r
        N.call("hsd_mamba_select_row", N.ptr(cb.cur), None, n, n, 4, None, N.stream(dev))
    d = (cur0 + V) % 4
    assert int(cb.cur.item()) == d and int(ca.cur.item()) == cur0
    assert torch.equal(ca.ssm[d].view(torch.int32), cb.ssm[d].view(torch.int32))
    assert torch.equal(ca.conv[d].view(torch.int16), cb.conv[d].view(torch.int16))


@pytest.mark.parametrize("T,pos0,total", [(1, 0, 1), (31, 0, 31), (33, 0, 33), (65, 0, 65), (130, 7, 137), (70, 100, 160)])
def test_attention(dev, T, pos0, total):
    HQ, HKV, HD, smax = 8, 2, 128, 192
    g = gen(dev, T)
    qkv = torch.randn((T, (HQ + 2 * HKV) * HD), device=dev, generator=g).to(torch.bfloat16)
    kv = nn.KVCache(HKV, smax, dev, HD)
    for t in (kv.k, kv.v):
        t[:, :pos0] = torch.randn((HKV, pos0, HD), device=dev, generator=g).to(torch.bfloat16)
    kv.v[:, total:] = float("nan")           # never read
    pos = torch.full((1,), pos0, dtype=torch.int32, device=dev)
    o = chunk.attention(qkv, kv, pos, total, n_heads=HQ, n_kv_heads=HKV, head_dim=HD)
    V = min(total - pos0, T)
    k, v = (qkv[:V, (HQ + i * HKV) * HD:(HQ + (i + 1) * HKV) * HD].view(V, HKV, HD).transpose(0, 1) for i in (0, 1))
    assert torch.equal(kv.k[:, pos0:pos0 + V].view(torch.int16), k.contiguous().view(torch.int16))
    assert torch.equal(kv.v[:, pos0:pos0 + V].view(torch.int16), v.contiguous().view(torch.int16))
    assert bool(torch.isnan(kv.v[:, total:].float()).all())
    q = qkv[:V, :HQ * HD].view(V, HQ, HD).double().cpu()
    kd, vd = kv.k.double().cpu(), kv.v.double().cpu()
    for r in (0, V // 2, V - 1):
        n = pos0 + r + 1
        for h in range(HQ):
            s = (kd[h // (HQ // HKV), :n] @ q[r, h]) / math.sqrt(HD)
            ref = torch.softmax(s, 0) @ vd[h // (HQ // HKV), :n]
            got = o[r, h * HD:(h + 1) * HD].double().cpu()
            assert float(((got - ref).abs() - 2.0 ** -8 * ref.abs()).max()) <= 2.0 ** -15 * 8, (r, h)


def test_attention_refuses_overflow(dev):
    HQ, HKV, HD, smax = 8, 2, 128, 64
    qkv = torch.ones((40, (HQ + 2 * HKV) * HD), dtype=torch.bfloat16, device=dev)
    kv = nn.KVCache(HKV, smax, dev, HD)
    status = torch.zeros(1, dtype=torch.int32, device=dev)
    pos = torch.full((1,), 30, dtype=torch.int32, device=dev)
    o = chunk.attention(qkv, kv, pos, 70, n_heads=HQ, n_kv_heads=HKV, head_dim=HD, status=status)
    assert int(status.item()) == N.STATUS_BAD_STATE
    assert float(kv.k.float().abs().max()) == 0 and float(o.float().abs().max()) == 0


@pytest.mark.parametrize("T,pos0,row", [(40, 0, 39), (70, 0, 33), (70, 5, 64), (130, 100, 0), (64, 0, 63)])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_attention_is_causal_for_values_that_are_not_finite(dev, T, pos0, row, value):
    """One value of row `row` is infinite or NaN: the rows ahead of it are bit for bit what they
    are without it, and so is every other dimension behind it; that one is not finite there."""
    HQ, HKV, HD, smax = 8, 2, 128, 256
    g = gen(dev, T)
    qkv = torch.randn((T, (HQ + 2 * HKV) * HD), device=dev, generator=g).to(torch.bfloat16)
    old = torch.randn((2, HKV, pos0, HD), device=dev, generator=g).to(torch.bfloat16)
    dim = 77
    odd = qkv.clone()
    odd[row, (HQ + HKV) * HD + dim] = value          # kv head 0
    out = []
    for x in (qkv, odd):
        kv = nn.KVCache(HKV, smax, dev, HD)
        kv.k[:, :pos0], kv.v[:, :pos0] = old[0], old[1]
        pos = torch.full((1,), pos0, dtype=torch.int32, device=dev)
        out.append(chunk.attention(x, kv, pos, pos0 + T, n_heads=HQ, n_kv_heads=HKV, head_dim=HD).view(T, HQ, HD))
    a, b = out
    keep = torch.ones((T, HQ, HD), dtype=torch.bool, device=dev)
    keep[row:, :HQ // HKV, dim] = False
    assert torch.equal(a.view(torch.int16)[keep], b.view(torch.int16)[keep])
    assert not bool(torch.isfinite(b.float())[~keep].any())


CFG = Mdl.ModelConfig(hidden=512, pattern="MEM*EME", vocab=4096, n_experts=16, topk=6, moe_inter=256, shared_inter=512,
                      max_seq=256, mtp=True)


@pytest.mark.parametrize("T", [4, 33, 70])
def test_chunked_prefill(dev, T):
    m = Mdl.NemotronModel(CFG, seed=5, device=dev, calibrate=False)
    prompt = np.random.default_rng(T).integers(0, CFG.vocab, T).astype(np.int32)
    caches, xs = [], []
    for mode, steps in (("sparse", False), ("dense", False), ("sparse", True)):
        m.set_mode(mode)
        m._chunkable = (lambda: False) if steps else (lambda: True)
        c = m.make_cache(cap=8)
        xs.append(m.prefill(prompt, c, graph=False).clone())
        assert int(c.status.item()) == 0
        caches.append(c)
    a, b, s = caches
    assert torch.equal(xs[0].view(torch.int16), xs[1].view(torch.int16))
    assert torch.equal(a.seq, b.seq) and torch.equal(a.seq, s.seq)
    assert a.state()[N.SEQ_POS] == T and a.state()[N.SEQ_HEAD_POS] == T - 1
    cur = int(a.cur.item())
    tensors = lambda c: [t for lc in c.layers if lc is not None for t in                          # noqa: E731
                         ((lc.ssm[cur], lc.conv[cur]) if hasattr(lc, "ssm") else (lc.k[:, :T], lc.v[:, :T]))] + \
        [c.head_kv.k[:, :T - 1], c.head_kv.v[:, :T - 1]]
    for u, v, w in zip(tensors(a), tensors(b), tensors(s)):
        assert torch.equal(u, v)
        u, w = u.double(), w.double()
        assert float((u - w).norm() / w.norm()) < 0.12 / math.sqrt(T) + 2e-2
    assert float((xs[0].double() - xs[2].double()).norm() / xs[2].double().norm()) < 0.24 + 2e-2   # one row


def off_by_one(t):
    """t at an address that is no multiple of 16 bytes."""
    return torch.zeros(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape).copy_(t)


class OwnRows(Mdl.MambaBlock):
    pass


@pytest.mark.parametrize("change", ["none", "pw", "head spw", "conv_w", "conv_b", "class", "eh_proj"])
def test_which_models_run_in_chunks(dev, change):
    """The unpatched rule takes this configuration; weights that the chunk kernels' loads or
    products do not take, and blocks of other classes, run in steps of 3 rows; a 4-bit eh_proj
    (1024 inputs) runs in chunks."""
    m = Mdl.NemotronModel(CFG, seed=5, device=dev, calibrate=False)
    prompt = np.random.default_rng(7).integers(0, CFG.vocab, 20).astype(np.int32)
    mamba, moe = m.blocks[0], m.blocks[1]
    if change == "pw":
        moe.pw = off_by_one(moe.pw)
    elif change == "head spw":
        m.mtp.moe.spw = off_by_one(m.mtp.moe.spw)
    elif change in ("conv_w", "conv_b"):
        setattr(mamba.mixer, change, off_by_one(getattr(mamba.mixer, change)))
    elif change == "class":
        mamba.__class__ = OwnRows
    elif change == "eh_proj":
        w = m.mtp.eh_proj
        m.mtp.eh_proj = nn.QWeight(*Mdl._Init(3, dev).q4(w.O, w.I, 1.0 / math.sqrt(w.I)))
    chunks = change in ("none", "eh_proj")
    assert m._chunkable() is chunks
    a, b = m.make_cache(cap=8), m.make_cache(cap=8)
    xa = m.prefill(prompt, a, graph=False).clone()
    m._chunkable = lambda: False
    xb = m.prefill(prompt, b, graph=False).clone()
    assert int(a.status.item()) == 0 and torch.equal(a.seq, b.seq)
    n = prompt.size - 1
    for u, v in ((a.head_kv.k[:, :n], b.head_kv.k[:, :n]), (a.head_kv.v[:, :n], b.head_kv.v[:, :n]), (xa, xb)):
        if chunks:
            assert float((u.double() - v.double()).norm() / v.double().norm()) < 0.26      # as test_chunked_prefill
        else:
            assert torch.equal(u.contiguous().view(torch.int16), v.contiguous().view(torch.int16))


@pytest.mark.parametrize("rows,T", [(16, 33), (16, 70), (17, 35), (17, 70), (3, 8)])
def test_prompt_of_several_chunks(dev, rows, T, monkeypatch):
    """Conv window, recurrent state, earlier chunks' keys, token and head offsets across chunks,
    a last chunk of one row (for which the head has none) and chunks of a multiple of the ring's
    4 slabs (the state goes to the slab it came from): against one chunk and against steps of 3
    rows. Without MoE layers (no ties between experts) two correct runs differ by bf16 roundings
    alone: 2^-9 each, a dozen of them on a row's way through these layers, a few times that where
    a norm follows. A lost state, window or key changes rows by a tenth of their size or more.
    (A state is compared by heads: a state row is a sum of one channel's x times B, and a channel
    whose x cancels in the conv has an x of nothing but roundings.)"""
    cfg = Mdl.ModelConfig(hidden=512, pattern="M*MM*", vocab=4096, n_experts=16, topk=6, moe_inter=256, shared_inter=512,
                          max_seq=256, mtp=True)
    m = Mdl.NemotronModel(cfg, seed=5, device=dev, calibrate=False)
    prompt = np.random.default_rng(T).integers(0, cfg.vocab, T).astype(np.int32)
    runs = []
    for mode in ("chunks", "one", "steps"):
        monkeypatch.setattr(Mdl, "CHUNK_ROWS", rows if mode == "chunks" else 2048)
        if mode == "steps":
            m._chunkable = lambda: False
        c = m.make_cache(cap=8)
        x = m.prefill(prompt, c, graph=False).clone()
        assert int(c.status.item()) == 0
        assert c.state()[N.SEQ_POS] == T and c.state()[N.SEQ_HEAD_POS] == T - 1
        cur = int(c.cur.item())
        t = [x[0]] + [r for lc in c.layers for r in ((lc.ssm[cur].flatten(1), lc.conv[cur]) if hasattr(lc, "ssm") else
                                                     (lc.k[:, :T], lc.v[:, :T]))]
        assert not bool(c.head_kv.k[:, T - 1:].any()) or mode == "steps"
        runs.append((cur, t + [c.head_kv.k[:, :T - 1], c.head_kv.v[:, :T - 1]]))
    assert runs[0][0] == runs[1][0] == runs[2][0] == T % 4
    for other in runs[1:]:
        for i, (u, v) in enumerate(zip(runs[0][1], other[1])):
            u, v = u.double(), v.double()
            err = (u - v).norm(dim=-1) / v.norm(dim=-1).clamp_min(1e-3 * float(v.norm(dim=-1).max()))
            assert float(err.max()) < 0.04, (i, float(err.max()))


@pytest.mark.parametrize("T", [5, 33, 100])
def test_blocks_on_the_same_rows(dev, T):
    """Each block of the model on the same input rows, as a chunk and in steps of 3 rows: one
    layer's roundings (2^-9 of a row's update, two or three of them, against the update itself);
    MoE rows but the few whose last expert is nearly tied. 100 rows: 64-slot tiles (100 * 6 >= 32
    * 16)."""
    m = Mdl.NemotronModel(CFG, seed=5, device=dev, calibrate=False)
    g = gen(dev, T)
    x = torch.randn((T, CFG.hidden), device=dev, generator=g).to(torch.bfloat16)
    x[:, 0] = m.c0
    for t, blk in zip(CFG.pattern[:4], m.blocks):
        a, b = m.make_cache(cap=8), m.make_cache(cap=8)
        li = CFG.pattern.index(t)
        u, v = x.clone(), x.clone()
        if t == "E":
            blk.chunk(u)
        else:
            blk.chunk(u, a.layers[li], a.pos, T, status=a.status)
        buf = m._bufs[3]
        for r in range(0, T, 3):
            n = min(3, T - r)
            if t == "E":
                blk.rows(v[r:r + n], buf)
                continue
            if t == "M":
                blk.rows(v[r:r + n], buf, b.layers[li], status=b.status)
                N.call("hsd_mamba_select_row", b.cur, None, n, n, Mdl.NSLAB, None, N.stream(dev))
            else:
                blk.rows(v[r:r + n], buf, b.layers[li], b.pos, status=b.status)
            N.call("hsd_seq_add", b.seq, N.SEQ_POS, n, N.stream(dev))
        step = (v.double() - x.double()).norm(dim=-1)
        err = (u.double() - v.double()).norm(dim=-1) / step
        far = err > 0.03
        assert float(far.double().mean()) <= (0.05 if t == "E" else 0.0), (t, float(err.max()))
        assert int(a.status.item()) == 0 and int(b.status.item()) == 0

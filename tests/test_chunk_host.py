"""CPU: what the MoE block's prompt path refuses before any launch: its kernels take rows of
hidden bf16 values, and read whatever they are given as such."""
import pytest
import torch

from hsd import _native as N
from hsd import chunk, mamba, nn
from hsd import model as Mdl


@pytest.mark.parametrize("rows,shape,dtype,tt", [
    (5, (5, 2688), torch.float16, 32), (64, (64, 2688), torch.float32, 32), (5, (5, 2560), torch.bfloat16, 32),
    (5, (5, 1, 2688), torch.bfloat16, 32), (5, (5, 2688), torch.bfloat16, 16), (5, (5, 2688), torch.bfloat16, 0),
    (2, (2, 2688), torch.float16, 32), (64, (64, 2688), torch.bfloat16, 48)])
def test_prefill_refuses(rows, shape, dtype, tt):
    blk = Mdl.MoEBlock.__new__(Mdl.MoEBlock)
    blk.cfg = Mdl.ModelConfig()
    assert blk.cfg.hidden == 2688
    with pytest.raises(N.HSDError, match="bf16 rows of 2688|slots"):
        blk.prefill_sparse(torch.zeros(shape, dtype=dtype), tt)


def test_products_refuse():
    """What nn.linear and mamba.ssm_rows refuse: another width (the kernels would read past the
    rows), another type or stride, and a residual that the product would not add."""
    bf = torch.bfloat16
    rows = chunk.Rows(torch.zeros((5, 128), dtype=bf), torch.zeros((5, 24), dtype=bf))
    q4 = nn.QWeight(torch.zeros((64, 16), dtype=torch.int32), torch.zeros((64, 2), dtype=bf), torch.zeros((64, 2), dtype=bf))
    wide = nn.QWeight(torch.zeros((64, 32), dtype=torch.int32), torch.zeros((64, 4), dtype=bf), torch.zeros((64, 4), dtype=bf))
    dense = nn.QWeight(torch.zeros((64, 128), dtype=bf))
    y = torch.zeros((5, 64), dtype=bf)
    bad = [(lambda: chunk.gemm(rows, wide), "128 inputs"),
           (lambda: chunk.gemm(rows, nn.QWeight(torch.zeros((64, 136), dtype=bf))), "128 inputs"),
           (lambda: chunk.gemm(chunk.Rows(rows.xp, None), q4), "group sums"),
           (lambda: chunk.gemm(rows, dense, residual=y), "residual"),
           (lambda: chunk.gemm(rows, q4, residual=y.float()), "bf16 rows"),
           (lambda: chunk.gemm(rows, q4, residual=y[:4]), "bf16 rows"),
           (lambda: chunk.gemm(rows, q4, out=torch.zeros((64, 5), dtype=bf).t()), "bf16 rows"),
           (lambda: chunk.prep(rows.xp.float()), "bf16 rows"),
           (lambda: chunk.prep(torch.zeros((128, 5), dtype=bf).t()), "unit-stride"),
           (lambda: chunk.prep(torch.zeros((5, 544)), gated_z=True), "norm weight")]
    mixer = mamba.Mamba2Mixer(*[torch.zeros(1)] * 6, num_heads=2, head_dim=16, n_groups=1)
    bad += [(lambda: chunk.scan(mixer, torch.zeros((5, 321), dtype=bf), None, None, 5), "322 unit-stride"),
            (lambda: chunk.scan(mixer, torch.zeros((5, 322)), None, None, 5), "322 unit-stride")]
    for f, why in bad:
        with pytest.raises(N.HSDError, match=why):
            f()


def test_rows_per_call_stay_below_a_gib():
    for D, F, FS, k in ((2688, 1856, 3712, 6), (128, 64, 64, 1), (3072, 8192, 16384, 8)):
        T = chunk.moe_rows(D, F, FS, k)
        gp = chunk.group_pitch(max(F, FS))
        assert T >= 1 and T * max(2 * (k * F + FS), 6 * (k + 1) * gp, 4 * (k + 1) * D) < 1 << 30

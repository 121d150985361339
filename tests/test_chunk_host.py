"""CPU: what the MoE block's prompt path refuses before any launch: its kernels take rows of
hidden bf16 values, and read whatever they are given as such."""
import pytest
import torch

from hsd import _native as N
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


def test_rows_per_call_stay_below_a_gib():
    from hsd import chunk
    for D, F, FS, k in ((2688, 1856, 3712, 6), (128, 64, 64, 1), (3072, 8192, 16384, 8)):
        T = chunk.moe_rows(D, F, FS, k)
        gp = chunk.group_pitch(max(F, FS))
        assert T >= 1 and T * max(2 * (k * F + FS), 6 * (k + 1) * gp, 4 * (k + 1) * D) < 1 << 30

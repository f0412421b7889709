"""The one-row q5_K / q6_K GEMV with several weight rows to a wave (gemv_k1_kernel): last rounds of rows that are full, nearly
empty and odd, rows of fewer super-blocks than a pass. Bit for bit the one-row-a-wave kernel's results, which products of
fewer rows run."""
import numpy as np
import pytest

import kungfu_amd as kf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ty,n", [(kf.TYPE_Q5_K, 2304), (kf.TYPE_Q5_K, 4096), (kf.TYPE_Q6_K, 4096)])
@pytest.mark.parametrize("n_out,bias,res", [(12288, True, True), (12289, False, True), (16383, True, False), (20481, False, False)])
def test_many_rows(cuda, ty, n, n_out, bias, res):
    import torch

    period = 509  # no multiple of a block's or the grid's rows
    w = kf.quantize(ty, kf.synth_normal(n, 0.02, period * n).reshape(period, n))
    wd = torch.from_numpy(w).to(cuda).repeat(-(-n_out // period), 1)[:n_out].contiguous()
    x = torch.from_numpy(kf.synth_normal(n + 1, 1.0, n).reshape(1, n)).to(cuda)
    b = torch.arange(n_out, device=cuda, dtype=torch.float32) if bias else None
    r = torch.arange(n_out, device=cuda, dtype=torch.float32).mul(0.5).view(1, -1) if res else None
    act, y = kf.alloc_act(1, n, cuda), torch.full((1, n_out), float("nan"), device=cuda)
    kf.matmul(ty, wd, x, act, y, n_out, bias=b, res=r)
    want = torch.empty(1, n_out, device=cuda)
    for a in range(0, n_out, 8000):
        e = min(a + 8000, n_out)
        part = torch.full((1, e - a), float("nan"), device=cuda)
        kf.matmul(ty, wd[a:e].clone(), x, act, part, e - a, bias=None if b is None else b[a:e].clone(), res=None if r is None else r[:, a:e].clone())
        want[:, a:e] = part
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy(), want.cpu().numpy())

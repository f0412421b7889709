"""One-row q8_0 products whose rows are not 16-byte aligned (a number of blocks that is no multiple of eight) run the pipelined
GEMV and quantize, or normalise, their activation row in it: bit for bit the two-launch result, and the CPU backend's."""
import numpy as np
import pytest

import kungfu_amd as kf
import oracle

pytestmark = pytest.mark.gpu
TY = kf.TYPE_Q8_0


@pytest.mark.parametrize("n,n_out", [(32, 1), (96, 5), (288, 640), (1056, 353), (4064, 2051), (6176, 700), (16352, 33)])
def test_ragged_rows(cuda, knobs, n, n_out):
    import torch

    dev = cuda
    w = kf.quantize(TY, kf.synth_normal(n, 0.02, n_out * n).reshape(n_out, n))
    x = kf.synth_normal(n + 1, 1.0, n).reshape(1, n)
    bias, res = kf.synth_normal(3, 1.0, n_out), kf.synth_normal(4, 1.0, n_out).reshape(1, n_out)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    wd, xd, bd, rd, nw = t(w), t(x), t(bias), t(res), t(np.abs(x[0]) + 0.5)
    act = kf.alloc_act(1, n, dev)
    parts = [(0, n_out // 3 + 1), (n_out // 3 + 1, n_out)] if n_out > 2 else [(0, n_out)]
    # a weight base is 16-byte aligned, so the group's members are copies of their own
    mw = [wd[a:b].clone() for a, b in parts]

    def run():
        y = [torch.full((1, n_out), float("nan"), device=dev) for _ in range(3)]
        kf.matmul(TY, wd, xd, act, y[0], n_out, bias=bd, res=rd)
        kf.rms_norm_matmul(TY, wd, xd, act, y[1], n_out, norm_w=nw, norm_b=nw)
        ys = [torch.full((1, b - a), float("nan"), device=dev) for a, b in parts]
        kf.matmul_group(TY, [(m, o, bd[a:b].clone(), None) for m, o, (a, b) in zip(mw, ys, parts)], xd, act)
        kf.quant_act(xd, act, kf.ACT_Q8_0)
        kf.gemv(TY, wd, act, y[2], 1, n, n_out)
        torch.cuda.synchronize()
        return [o.cpu().numpy() for o in y + ys]

    got = run()
    knobs.setenv("KF_MATMUL_NO_FUSE", 1)
    knobs.setenv("KF_GEMV_NO_DMA", 1)
    for a, b in zip(got, run()):
        assert np.array_equal(a, b)
    # one f32 rounding (2^-24) of a partial sum of magnitude below 16 a group, on either side
    err = np.abs(got[0].astype(np.float64) - (oracle.matmul_i8(TY, w, n, n_out, x, bias) + res))
    assert err.max() <= 2 * (n // 32 + 2) * 2.0**-24 * 16

"""The q8_0 tile GEMM of any width (gemm_q8.hip) at the sizes where its tiling can go wrong: widths of one block, of an odd
number of blocks (rows that start at every even byte of a 16-byte piece), around the 128-column stage, row counts around the
32-, 64- and 128-row tiles, output columns around the 256-column tile, split and unsplit, through the entry points
that take it. Against the CPU backend's int8 path: the same integers, f32 sums of at most 448 terms in another order."""
import numpy as np
import pytest

import kungfu_amd as kf
import oracle

pytestmark = pytest.mark.gpu
TY = kf.TYPE_Q8_0


def _t(a, dev):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _blocks(n_out, n, seed):
    return kf.quantize(TY, kf.synth_normal(seed, 0.02, n_out * n).reshape(n_out, n))


def _close(got, want, n):
    # one f32 rounding (2^-24) of a partial sum of magnitude below 16 a group, on either side
    err = np.abs(got.astype(np.float64) - want.astype(np.float64))
    assert err.max() <= 2 * (n // 32 + 2) * 2.0**-24 * 16, f"max err {err.max():.3e}"


@pytest.mark.parametrize("v", [0, 1, 2])
@pytest.mark.parametrize("rows,n,n_out", [(2, 32, 1), (31, 96, 255), (33, 128, 257), (65, 160, 40), (129, 1056, 300), (64, 2080, 33),
                                          (128, 4128, 256), (9, 14336, 70), (40, 256, 513)])
def test_tile_edges(cuda, knobs, v, rows, n, n_out):
    import torch

    w = _blocks(n_out, n, rows + n + n_out)
    x = kf.synth_normal(rows + n, 1.0, rows * n).reshape(rows, n)
    bias, res = kf.synth_normal(3, 1.0, n_out), kf.synth_normal(4, 1.0, rows * n_out).reshape(rows, n_out)
    want = oracle.matmul_i8(TY, w, n, n_out, x, bias) + res
    knobs.setenv("KF_Q8_V", v)
    # infinite and NaN scales around the matrix: a read past its rows or columns that counted would meet them
    wt = torch.full((w.size + 4096,), 0x7C, dtype=torch.uint8, device=cuda)
    wt[: w.size] = _t(w.reshape(-1), cuda)
    act = kf.alloc_act(rows, n, cuda)
    act.fill_(0xFF)
    kf.quant_act(_t(x, cuda), act, kf.ACT_Q8_0)
    args = dict(bias=_t(bias, cuda), res=_t(res, cuda))
    got = []
    for call in (kf.gemv, kf.gemv) + ((kf.gemm_i8,) if n % 128 == 0 else ()):
        y = torch.full((rows, n_out), float("nan"), device=cuda)
        call(TY, wt, act, y, rows, n, n_out, **args)
        torch.cuda.synchronize()
        got.append(y.cpu().numpy())
    _close(got[0], want, n)
    for g in got[1:]:
        assert np.array_equal(got[0].view(np.uint32), g.view(np.uint32))
    knobs.setenv("KF_GEMM_NO_TAIL", 1)
    kf.gemv(TY, wt, act, y, rows, n, n_out, **args)
    torch.cuda.synchronize()
    _close(y.cpu().numpy(), want, n)


@pytest.mark.parametrize("rows,n,n_out", [(3, 1056, 300), (20, 1056, 300), (300, 1248, 700), (90, 2176, 600), (17, 9248, 100)])
def test_matmul_takes_any_width(cuda, rows, n, n_out):
    import torch

    w = _blocks(n_out, n, rows + n)
    x = kf.synth_normal(rows, 1.0, rows * n).reshape(rows, n)
    act = kf.alloc_act(rows, n, cuda)
    y = torch.full((rows, n_out), float("nan"), device=cuda)
    kf.matmul(TY, _t(w, cuda), _t(x, cuda), act, y, n_out)
    torch.cuda.synchronize()
    _close(y.cpu().numpy(), oracle.matmul_i8(TY, w, n, n_out, x, None), n)


def test_infinite_activation_scale(cuda, knobs):
    """A group with an infinite activation has an infinite scale; the row's other columns and the other rows stay what
    they are, and the row is infinite or NaN where the CPU's is, as with the older kernel."""
    import torch

    rows, n, n_out = 33, 512, 40
    w = _blocks(n_out, n, 5)
    x = kf.synth_normal(6, 1.0, rows * n).reshape(rows, n)
    x[7, 100] = np.inf
    act = kf.alloc_act(rows, n, cuda)
    outs = []
    for v in (0, 3):
        knobs.setenv("KF_Q8_V", v)
        y = torch.full((rows, n_out), 0.5, device=cuda)
        kf.matmul(TY, _t(w, cuda), _t(x, cuda), act, y, n_out)
        torch.cuda.synchronize()
        outs.append(y.cpu().numpy())
    finite = np.arange(rows) != 7
    assert np.isfinite(outs[0][finite]).all() and not np.isfinite(outs[0][7]).any()
    assert np.array_equal(np.isfinite(outs[0]), np.isfinite(outs[1]))


@pytest.mark.parametrize("rows,n,n_out", [(2, 4064, 14000), (3, 4032, 9000), (5, 1056, 300), (8, 2336, 3001), (9, 2336, 726)])
def test_matmul_and_gemv_take_the_same_product(cuda, rows, n, n_out):
    """A few rows of a width that only kf_hip_gemv's rule covers: kf_hip_matmul, kf_hip_gemv and both group forms run the same
    kernel, bit for bit."""
    import torch

    w = _t(_blocks(n_out, n, rows + n), cuda)
    x = _t(kf.synth_normal(rows, 1.0, rows * n).reshape(rows, n), cuda)
    act = kf.alloc_act(rows, n, cuda)
    ys = [torch.full((rows, n_out), float("nan"), device=cuda) for _ in range(4)]
    kf.matmul(TY, w, x, act, ys[0], n_out)
    kf.matmul_group(TY, [(w, ys[1], None, None)], x, act)
    kf.gemv(TY, w, act, ys[2], rows, n, n_out)
    kf.gemv_group(TY, [(w, ys[3], None, None)], act, rows, n)
    torch.cuda.synchronize()
    bits = [y.cpu().numpy().view(np.uint32) for y in ys]
    for b in bits[1:]:
        assert np.array_equal(bits[0], b)


def _exact(w, act, rows, n, n_out):
    """The product of the rows quantized in `act` with the weight bytes, in 64 bits."""
    offs, raw = kf.act_offsets(rows, n), act.cpu().numpy()
    xq = raw[offs[0] : offs[0] + rows * n].view(np.int8).reshape(rows, n // 32, 32).astype(np.float64)
    xd = raw[offs[3] : offs[3] + rows * n // 32 * 4].view(np.float32).reshape(rows, n // 32, 1).astype(np.float64)
    b = w.reshape(n_out, n // 32, 34)
    wd = np.ascontiguousarray(b[:, :, :2]).view(np.float16).astype(np.float64)
    wq = np.ascontiguousarray(b[:, :, 2:]).view(np.int8).astype(np.float64)
    return (xq * xd).reshape(rows, n) @ (wq * wd).reshape(n_out, n).T


@pytest.mark.parametrize("tail", [True, False])
@pytest.mark.parametrize("rows,n,n_out", [(3, 4032, 2000), (33, 2080, 1000), (20, 14048, 640), (300, 14368, 512), (700, 4128, 300)])
def test_ragged_widths_lose_no_precision(cuda, knobs, rows, n, n_out, tail):
    """Widths that are no multiple of 128 columns, with K split and whole: no further from the 64-bit product than the
    multi-row product, which sums over 64 lanes. Eight groups an f32 sum: the roundings of a partial sum of k of 8 equal
    terms, k = 2..8, and of the term itself, each of rms at most 2^-24 / sqrt(3) of the partial, make sqrt(5.4) of these."""
    import torch

    w = _blocks(n_out, n, rows + n)
    x = kf.synth_normal(rows, 1.0, rows * n).reshape(rows, n)
    act = kf.alloc_act(rows, n, cuda)
    kf.quant_act(_t(x, cuda), act, kf.ACT_Q8_0)
    want = _exact(w, act, rows, n, n_out)
    if not tail:
        knobs.setenv("KF_GEMM_NO_TAIL", 1)
    errs = []
    # the product the cost picks, the 32- and 64-row tiles, the multi-row product
    for v in (None, 0, 1, 3):
        if v is not None:
            knobs.setenv("KF_Q8_V", v)
        y = torch.full((rows, n_out), float("nan"), device=cuda)
        kf.matmul(TY, _t(w, cuda), _t(x, cuda), act, y, n_out)
        torch.cuda.synchronize()
        errs.append(np.linalg.norm(y.cpu().numpy() - want) / np.linalg.norm(want))
    assert max(errs[:3]) <= errs[3] and max(errs[1:3]) <= np.sqrt(5.4) * 2.0**-24 / np.sqrt(3), errs


def test_small_matrices_keep_the_small_batch_kernels(cuda, knobs):
    """48 rows of 1024 -> 512: the small-batch kernels' bits (KF_Q8_V=3), not the tile GEMM's, which takes longer there."""
    import torch

    rows, n, n_out = 48, 1024, 512
    w = _t(_blocks(n_out, n, 9), cuda)
    x = _t(kf.synth_normal(rows, 1.0, rows * n).reshape(rows, n), cuda)
    act = kf.alloc_act(rows, n, cuda)
    bits = []
    for v in (None, 3, 0):
        if v is not None:
            knobs.setenv("KF_Q8_V", v)
        y = torch.full((rows, n_out), float("nan"), device=cuda)
        kf.matmul(TY, w, x, act, y, n_out)
        torch.cuda.synchronize()
        bits.append(y.cpu().numpy().view(np.uint32))
    assert np.array_equal(bits[0], bits[1]) and not np.array_equal(bits[0], bits[2])

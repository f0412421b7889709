"""The K-quant tile GEMM (gemm_kq.hip) at the sizes where its tiling can go wrong: super-block counts that start q6_K rows
at every even byte offset, row counts around the 32-row tiles of a block, output columns around the 256-column tiles, split
and unsplit, and the grouped form's ranges over uneven slots. Outputs against the CPU backend's int8 path (the same
integers; the f32 sums of at most 56 super-blocks differ by their order only)."""
import numpy as np
import pytest

import kungfu_amd as kf
import oracle

pytestmark = pytest.mark.gpu
K_TYPES = [kf.TYPE_Q4_K, kf.TYPE_Q5_K, kf.TYPE_Q6_K]


def _t(a, dev):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _blocks(ty, n_out, n, seed):
    return kf.quantize(ty, kf.synth_normal(seed, 0.02, n_out * n).reshape(n_out, n))


def _close(got, want):
    # 2^-24 for each of a row's sums of up to 56 super-block terms of magnitude below 8
    err = np.abs(got.astype(np.float64) - want.astype(np.float64))
    assert err.max() <= 56 * 2.0**-24 * 8, f"max err {err.max():.3e}"


@pytest.mark.parametrize("tm", [1, 2, 4])
@pytest.mark.parametrize("ty", K_TYPES)
@pytest.mark.parametrize("rows,n,n_out", [(2, 256, 1), (31, 768, 255), (33, 1280, 257), (65, 1792, 40), (129, 2304, 300), (96, 2560, 33),
                                          (128, 3328, 256), (40, 14336, 70)])
def test_tile_edges(cuda, knobs, ty, tm, rows, n, n_out):
    import torch

    w = _blocks(ty, n_out, n, rows + n + n_out)
    x = kf.synth_normal(rows + n, 1.0, rows * n).reshape(rows, n)
    bias, res = kf.synth_normal(3, 1.0, n_out), kf.synth_normal(4, 1.0, rows * n_out).reshape(rows, n_out)
    want = oracle.matmul_i8(ty, w, n, n_out, x, bias) + res
    knobs.setenv("KF_KQ_GEMM", 1)
    knobs.setenv("KF_KQ_TM", tm)
    # a guard row behind the matrix: reads past its last 16-byte piece would meet it
    wt = torch.full((w.size + 4096,), 255, dtype=torch.uint8, device=cuda)
    wt[: w.size] = _t(w.reshape(-1), cuda)
    act = kf.alloc_act(rows, n, cuda)
    got = []
    for _ in range(2):
        y = torch.full((rows, n_out), float("nan"), device=cuda)
        kf.matmul(ty, wt, _t(x, cuda), act, y, n_out, bias=_t(bias, cuda), res=_t(res, cuda))
        torch.cuda.synchronize()
        got.append(y.cpu().numpy())
    _close(got[0], want)
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    knobs.setenv("KF_GEMM_NO_TAIL", 1)
    kf.matmul(ty, wt, _t(x, cuda), act, y, n_out, bias=_t(bias, cuda), res=_t(res, cuda))
    torch.cuda.synchronize()
    _close(y.cpu().numpy(), want)


@pytest.mark.parametrize("scratch", [True, False])
@pytest.mark.parametrize("tm", [1, 2, 4])
@pytest.mark.parametrize("counts", [(1,), (0, 33, 0, 128, 5), (97, 96, 95, 64, 1, 0, 0, 31), tuple((7 * i) % 41 for i in range(70))])
def test_grouped_ranges(cuda, knobs, counts, tm, scratch):
    """Slots of no, few and many rows (more than 64 of them: two steps of the slot search) cut into ranges that start and end
    inside tiles; the output rows through a permutation, and the two-matrix form's columns past the split."""
    import torch

    ty, n, half = kf.TYPE_Q4_K, 512, 256
    pairs, n_slots = sum(counts), len(counts)
    offs = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    wa, wb = (_blocks(ty, n_slots * half, n, s) for s in (11, 12))
    x = kf.synth_normal(pairs, 1.0, pairs * n).reshape(pairs, n)
    rows = np.random.default_rng(pairs).permutation(pairs).astype(np.int32)
    knobs.setenv("KF_KQ_TM", tm)
    # the tiles cut into ranges, or whole
    if scratch:
        knobs.setenv("KF_KQ_G", 256)
    else:
        knobs.setenv("KF_GEMM_NO_TAIL", 1)
    act = kf.alloc_act(pairs, n, cuda)
    kf.quant_act(_t(x, cuda), act, kf.ACT_Q8K)
    y = torch.full((pairs, 2 * half), float("nan"), device=cuda)
    kf.moe_gemm(ty, _t(wa, cuda), act, pairs, n, 2 * half, _t(offs, cuda), n_slots, y, half * kf.row_bytes(ty, n), w2=_t(wb, cuda), n_split=half,
                out_rows=_t(rows, cuda))
    torch.cuda.synchronize()
    got = y.cpu().numpy()[rows]
    for s in range(n_slots):
        r0, r1 = offs[s], offs[s + 1]
        if r1 > r0:
            for at, w in ((0, wa), (half, wb)):
                _close(got[r0:r1, at : at + half], oracle.matmul_i8(ty, w[s * half : (s + 1) * half], n, half, x[r0:r1], None))


def test_matmul_past_the_gemv_width(cuda):
    """q4_K rows wider than kf_hip_gemv takes: kf_hip_matmul runs them from 96 rows on, as the GEMM."""
    import torch

    ty, rows, n, n_out = kf.TYPE_Q4_K, 96, 33024, 40
    w = _blocks(ty, n_out, n, 21)
    x = kf.synth_normal(22, 0.5, rows * n).reshape(rows, n)
    act = kf.alloc_act(rows, n, cuda)
    y = torch.full((rows, n_out), float("nan"), device=cuda)
    kf.matmul(ty, _t(w, cuda), _t(x, cuda), act, y, n_out)
    torch.cuda.synchronize()
    # 2^-24 for each of a row's sums of 129 super-block terms of magnitude below 16
    err = np.abs(y.cpu().numpy().astype(np.float64) - oracle.matmul_i8(ty, w, n, n_out, x, None))
    assert err.max() <= 2 * 129 * 2.0**-24 * 16
    with pytest.raises(kf.KfError):
        kf.matmul(ty, _t(w, cuda), _t(x[:95], cuda), act, y[:95], n_out)


@pytest.mark.parametrize("rows,n,n_out", [(40, 6400, 600), (300, 13056, 512), (700, 6400, 2304), (2048, 6400, 300)])
def test_ragged_q6_K_loses_no_precision(cuda, knobs, rows, n, n_out):
    """q6_K rows of an odd number of super-blocks: no further from the 64-bit product than the per-lane product, which sums
    over 64 lanes, by the plan and on 32- and 64-row tiles run whole. These sum in 64 bits: three roundings a super-block's
    term (its integer, the two scales) and the last one, each of rms at most 2^-24 / sqrt(3)."""
    import torch

    ty = kf.TYPE_Q6_K
    w = _blocks(ty, n_out, n, rows + n)
    x = kf.synth_normal(rows, 1.0, rows * n).reshape(rows, n)
    act = kf.alloc_act(rows, n, cuda)
    kf.quant_act(_t(x, cuda), act, kf.ACT_Q8K)
    offs, raw = kf.act_offsets(rows, n), act.cpu().numpy()
    xq = raw[offs[0] : offs[0] + rows * n].view(np.int8).reshape(rows, n // 32, 32).astype(np.float64)
    xd = raw[offs[3] : offs[3] + rows * n // 32 * 4].view(np.float32).reshape(rows, n // 32, 1).astype(np.float64)
    # q6_K weights are exact in f32: 11 bits of d, 7 of the scale, 6 of the value
    want = (xq * xd).reshape(rows, n) @ np.asarray(oracle.dequant(ty, w, n)).reshape(n_out, n).astype(np.float64).T
    errs = []
    for ks in ({"KF_KQ_GEMM": 0}, {}, {"KF_KQ_GEMM": 1, "KF_KQ_TM": 1, "KF_GEMM_NO_TAIL": 1}, {"KF_KQ_GEMM": 1, "KF_KQ_TM": 2, "KF_GEMM_NO_TAIL": 1}):
        for k, v in ks.items():
            knobs.setenv(k, v)
        y = torch.full((rows, n_out), float("nan"), device=cuda)
        kf.matmul(ty, _t(w, cuda), _t(x, cuda), act, y, n_out)
        torch.cuda.synchronize()
        errs.append(np.linalg.norm(y.cpu().numpy() - want) / np.linalg.norm(want))
        for k in ks:
            knobs.delenv(k)
    assert max(errs[1:]) <= errs[0] and max(errs[2:]) <= 2.0**-23 / np.sqrt(3), errs


@pytest.mark.parametrize("tail", [True, False])
@pytest.mark.parametrize("tm", [1, 2, 4])
@pytest.mark.parametrize("ty", K_TYPES)
def test_infinite_and_nan_block_scales(cuda, knobs, ty, tm, tail):
    """A super-block whose scale is infinite or NaN (and, of q4_K / q5_K, its minimum's): its output column is infinite or
    NaN as the CPU's is, and the other columns are those of the same matrix with finite scales, bit for bit."""
    import torch

    rows, n, n_out = 33, 4096, 300
    w = _blocks(ty, n_out, n, 31).reshape(n_out, n // 256, -1)
    bad = w.copy()
    at = (208,) if ty == kf.TYPE_Q6_K else (0, 2)
    for k, (row, sb, bits) in enumerate(((0, 0, 0x7C00), (31, 15, 0x7E00), (32, 7, 0xFC00), (255, 8, 0x7C00), (299, 3, 0x7E00))):
        bad[row, sb, at[k % len(at)] : at[k % len(at)] + 2] = np.array([bits], np.uint16).view(np.uint8)
    cols = [0, 31, 32, 255, 299]
    x = kf.synth_normal(32, 1.0, rows * n).reshape(rows, n)
    knobs.setenv("KF_KQ_GEMM", 1)
    knobs.setenv("KF_KQ_TM", tm)
    if not tail:
        knobs.setenv("KF_GEMM_NO_TAIL", 1)
    act = kf.alloc_act(rows, n, cuda)
    outs = []
    for m in (w, bad):
        y = torch.full((rows, n_out), 0.5, device=cuda)
        kf.matmul(ty, _t(m.reshape(n_out, -1), cuda), _t(x, cuda), act, y, n_out)
        torch.cuda.synchronize()
        outs.append(y.cpu().numpy())
    rest = np.setdiff1d(np.arange(n_out), cols)
    assert np.isfinite(outs[0]).all()
    assert np.array_equal(outs[0][:, rest].view(np.uint32), outs[1][:, rest].view(np.uint32))
    with np.errstate(all="ignore"):
        want = oracle.matmul_i8(ty, np.ascontiguousarray(bad[cols]).reshape(len(cols), -1), n, len(cols), x, None)
    # (which of the two, and an infinity's sign, follow the order of the terms; the CPU multiplies the scales out first)
    assert not np.isfinite(want).any() and not np.isfinite(outs[1][:, cols]).any()


@pytest.mark.parametrize("ty", K_TYPES)
@pytest.mark.parametrize("rows,n,n_out,gemm", [(300, 1024, 512, True), (256, 14336, 40, True), (200, 1792, 600, True), (48, 1024, 512, False), (96, 4096, 4352, True)])
def test_few_outputs_price_the_few_row_products_latency(cuda, knobs, ty, rows, n, n_out, gemm):
    """Matrices of few outputs: each 16-row pass of the few-row product costs the latency of a whole row, so many rows take
    the tile GEMM (the bits of KF_KQ_GEMM=1) and 48 short ones do not (those of KF_KQ_GEMM=0). So do 96 rows of 272 tiles, two
    a block on half the CUs."""
    import torch

    w = _t(_blocks(ty, n_out, n, rows + n), cuda)
    x = _t(kf.synth_normal(rows, 1.0, rows * n).reshape(rows, n), cuda)
    act = kf.alloc_act(rows, n, cuda)
    bits = []
    for force in (None, 0, 1):
        if force is not None:
            knobs.setenv("KF_KQ_GEMM", force)
        y = torch.full((rows, n_out), float("nan"), device=cuda)
        kf.matmul(ty, w, x, act, y, n_out)
        torch.cuda.synchronize()
        bits.append(y.cpu().numpy().view(np.uint32))
    assert not np.array_equal(bits[1], bits[2])
    assert np.array_equal(bits[0], bits[2 if gemm else 1])


@pytest.mark.parametrize("ty,rows,n,n_out,gemm", [(kf.TYPE_Q4_K, 16, 4608, 27648, False), (kf.TYPE_Q4_K, 25, 4608, 27648, True),
                                                  (kf.TYPE_Q4_K, 32, 8192, 16384, True), (kf.TYPE_Q5_K, 32, 4096, 28672, True),
                                                  (kf.TYPE_Q6_K, 28, 4096, 28672, True), (kf.TYPE_Q6_K, 17, 4096, 28672, False)])
def test_decoded_batches_keep_their_product(cuda, knobs, ty, rows, n, n_out, gemm):
    """Up to 32 rows kf_hip_matmul takes the tile GEMM on the largest matrices only, with K in two or four f32 ranges summed in
    order (the bits of a 128- or 64-row tile's plan as well), the few-row product elsewhere; kf_hip_gemv always the latter."""
    import torch

    w = _t(np.tile(_blocks(ty, 512, n, rows + n), (n_out // 512, 1)), cuda)
    x = _t(kf.synth_normal(rows, 1.0, rows * n).reshape(rows, n), cuda)
    act = kf.alloc_act(rows, n, cuda)
    kf.quant_act(x, act, kf.ACT_Q8K)

    def bits(entry, **ks):
        for k, v in ks.items():
            knobs.setenv(k, v)
        y = torch.full((rows, n_out), float("nan"), device=cuda)
        entry(y)
        torch.cuda.synchronize()
        for k in ks:
            knobs.delenv(k)
        return y.cpu().numpy().view(np.uint32)

    def matmul(y):
        kf.matmul(ty, w, x, act, y, n_out)

    def gemv(y):
        kf.gemv(ty, w, act, y, rows, n, n_out)

    few = bits(gemv, KF_KQ_GEMM=0)
    tiles = [bits(matmul, KF_KQ_GEMM=1, KF_KQ_TM=tm) for tm in (1, 2, 4)]
    assert np.array_equal(tiles[0], tiles[1]) and np.array_equal(tiles[0], tiles[2])
    assert not np.array_equal(few, tiles[0])
    assert np.array_equal(bits(matmul), tiles[0] if gemm else few)
    assert np.array_equal(bits(gemv), few)


@pytest.mark.parametrize("n_slots,pairs,n,n_out,cut", [(8, 209, 1280, 1536, False), (16, 110, 1280, 1536, False),
                                                       (8, 1024, 14336, 4096, True), (8, 128, 4096, 4096, True)])
def test_grouped_tiles_are_cut_where_that_pays(cuda, knobs, n_slots, pairs, n, n_out, cut):
    """Small experts run a block a tile (the bits of KF_GEMM_NO_TAIL), large ones in equal ranges (those of KF_KQ_G)."""
    import torch

    ty = kf.TYPE_Q4_K
    w = _t(np.tile(_blocks(ty, 512, n, pairs), (n_slots * n_out // 512, 1)), cuda)
    cnt = np.random.default_rng(1).multinomial(pairs, [1 / n_slots] * n_slots)
    offs = _t(np.concatenate([[0], np.cumsum(cnt)]).astype(np.int32), cuda)
    act = kf.alloc_act(pairs, n, cuda)
    kf.quant_act(_t(kf.synth_normal(pairs, 1.0, pairs * n).reshape(pairs, n), cuda), act, kf.ACT_Q8K)
    bits = []
    for name, value in ((None, None), ("KF_GEMM_NO_TAIL", 1), ("KF_KQ_G", 256)):
        if name:
            knobs.setenv(name, value)
        y = torch.full((pairs, n_out), float("nan"), device=cuda)
        kf.moe_gemm(ty, w, act, pairs, n, n_out, offs, n_slots, y, n_out * kf.row_bytes(ty, n))
        torch.cuda.synchronize()
        bits.append(y.cpu().numpy().view(np.uint32))
        if name:
            knobs.delenv(name)
    assert not np.array_equal(bits[1], bits[2])
    assert np.array_equal(bits[0], bits[2 if cut else 1])

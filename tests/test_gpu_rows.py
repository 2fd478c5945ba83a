"""GPU parity of vq_rows_gemm (vq2_rows_gemm: rotate any number of rows, pack
them, multiply by up to 4 VQ matrices on the matrix cores) against the fp64
oracle: edges of the 16-row, 16-column and 256-k tiles, workgroups that share
a tile's k tiles, every cfg and type, rows without alignment, several matrices
a launch, a row with NaN, and a captured call.

Tolerance: the oracle is fed the activation as the kernel holds it (rotated in
fp32 by vq_rht, whose stages run in the same order, then rounded to fp16 under
a power-of-two scale per row), so what is left is the order of fp32 sums: 1e-5
of max |y| over at most 8192 terms (~1e-7 observed), plus the result type's
rounding."""
import numpy as np
import pytest
import torch

from act_rounding import fp16_row_scaled
from compressai_amd import kernels as K, synth
from compressai_amd.kernels import Vq2Error
from compressai_amd.runtime import PackedLinear, PackedProjections
from oracle import vq2_oracle as O

pytestmark = pytest.mark.gpu

TOL_SUM = 1e-5
EPS = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _books(seed, bpw, dtype):
    cb0 = synth.codebook(seed, dtype=dtype)
    return cb0, {2: None, 3: synth.codebook(seed + 1, rows=256, dtype=dtype),
                 4: synth.codebook(seed + 1, dtype=dtype)}[bpw]


def _on(dev, *ts):
    return [None if t is None else t.to(dev) for t in ts]


def _check(y, xr, m, cb0, cb1, rs=1.0):
    # codebooks that are not fp16 are rounded to fp16
    h0, h1 = cb0.half(), None if cb1 is None else cb1.half()
    _, ref = O.vq_gemv(fp16_row_scaled(xr), m["idx0"], m["idx1"], h0, h1, m["scale"], rs=rs)
    got = y.float().cpu().numpy()
    for b in range(got.shape[0]):
        bound = TOL_SUM * np.abs(ref[b]).max() + EPS[y.dtype] * np.abs(ref[b])
        assert np.all(np.abs(got[b] - ref[b]) <= bound), (b, np.abs(got[b] - ref[b]).max())


@pytest.mark.parametrize("M,rows,n,hb,bpw,x_dtype,cb_dtype,y_dtype", [
    (1, 16, 64, 64, 2, torch.float32, torch.float16, torch.float32),        # two k blocks of one tile
    (3, 1, 320, 64, 4, torch.float16, torch.float16, torch.float32),        # 40 groups: a short second tile
    (16, 15, 512, 512, 3, torch.bfloat16, torch.bfloat16, torch.bfloat16),
    (17, 33, 2048, 2048, 2, torch.float16, torch.float32, torch.float16),
    (33, 100, 4096, 4096, 3, torch.float32, torch.float16, torch.float32),  # one exchange more
    (48, 47, 8192, 8192, 2, torch.float32, torch.float16, torch.float32),   # the widest row
    (49, 130, 5120, 1024, 4, torch.bfloat16, torch.float16, torch.float32),
    (64, 512, 6144, 2048, 4, torch.float16, torch.float16, torch.float16),  # four workgroups a tile
    (65, 2048, 6144, 2048, 2, torch.float16, torch.bfloat16, torch.float32),  # row blocks of 64 and 1
    (100, 700, 2048, 2048, 4, torch.float16, torch.float16, torch.float32),
    # 128 and 256 rows a workgroup: remainders of the row and column blocks, a
    # short last k tile, k tiles in one, two and four shares (every plan of
    # either: test_rows_gemm_plans)
    (129, 5003, 576, 64, 2, torch.float16, torch.float16, torch.float16),
    (65, 6001, 2048, 2048, 2, torch.bfloat16, torch.float16, torch.float32),
    (65, 3100, 2048, 2048, 4, torch.bfloat16, torch.bfloat16, torch.float32),
    (270, 5003, 512, 512, 3, torch.float32, torch.float16, torch.float32),
    (400, 5003, 512, 512, 2, torch.float16, torch.float32, torch.float16),
    (193, 3100, 1024, 1024, 4, torch.float16, torch.float16, torch.float32),
    # codebooks rounded as gathered (bf16 from 9 rows on, with fewer steps in
    # flight from 33 on at 3 bpw; fp32 with one 16-bit stage), and fp32 ones
    # of two such stages or more than 2^20 gathers
    (8, 77, 320, 64, 3, torch.float16, torch.bfloat16, torch.float32),
    (9, 77, 320, 64, 2, torch.float16, torch.bfloat16, torch.float32),
    (20, 130, 2048, 2048, 4, torch.bfloat16, torch.bfloat16, torch.bfloat16),
    (33, 65, 1024, 1024, 3, torch.float16, torch.bfloat16, torch.float32),
    (64, 33, 320, 64, 3, torch.float32, torch.bfloat16, torch.float32),
    (50, 600, 2048, 2048, 4, torch.float32, torch.bfloat16, torch.float32),
    (5, 700, 1024, 1024, 3, torch.float16, torch.float32, torch.float32),
    (40, 129, 320, 64, 2, torch.float32, torch.float32, torch.float32),
    (6, 129, 512, 512, 4, torch.float32, torch.float32, torch.float32),
    (3, 2200, 4096, 4096, 2, torch.float16, torch.float32, torch.float32),
])
def test_rows_gemm_vs_oracle(dev, M, rows, n, hb, bpw, x_dtype, cb_dtype, y_dtype):
    seed = 9900 + M
    m = synth.vq_matrix(seed, rows, n, bpw=bpw)
    cb0, cb1 = _books(seed + 1, bpw, cb_dtype)
    x = synth.activations(seed + 2, (M, n), dtype=x_dtype).to(dev)
    sign, perm = _on(dev, synth.signs(seed + 3, n), synth.permutation(seed + 4, n))
    mats = [tuple(_on(dev, m["idx0"], m["idx1"], m["scale"])) + (rows,)]
    c0, c1 = _on(dev, cb0, cb1)
    (y,) = K.vq_rows_gemm(x, mats, c0, c1, n, perm, sign, hb, out_dtype=y_dtype)
    xr = K.vq_rht(x, perm, sign, hb, out_dtype=torch.float32).cpu().numpy()
    _check(y, xr, m, cb0, cb1)
    if M > 128:
        return
    # no tables, then a rotated activation under another rs
    (y,) = K.vq_rows_gemm(x, mats, c0, c1, n, None, None, hb, out_dtype=y_dtype)
    _check(y, K.vq_rht(x, None, None, hb, out_dtype=torch.float32).cpu().numpy(), m, cb0, cb1)
    (y,) = K.vq_rows_gemm(x, mats, c0, c1, n, hb=0, rs=0.25, out_dtype=torch.float32)
    _check(y, x.float().cpu().numpy(), m, cb0, cb1, rs=0.25)


# The launch plans of 256 CUs (rows_plan), one case each: rows a workgroup,
# shares of the k tiles; column tiles a workgroup
@pytest.mark.parametrize("M,rows,n,bpw,cb_dtype", [
    # rows_wide_kernel, the last k tile short in all, shares of unequal k tiles in those of two or four
    (129, (6001,), 320, 2, torch.float16),               # 128 rows, 1 share
    (65, (6001,), 2240, 2, torch.float16),               # 2: 4 and 5 of 9 k tiles
    (65, (5003,), 3136, 3, torch.bfloat16),              # 4 of 13
    (65, (6001,), 1600, 4, torch.float16),               # 2 of 7
    (65, (3000,), 2240, 4, torch.float32),               # 4 of 9
    (129, (12300,), 320, 3, torch.float16),              # 256 rows, 1 share
    (129, (8200,), 2240, 3, torch.float16),              # 2 of 9
    (129, (3000,), 3136, 2, torch.bfloat16),             # 4 of 13
    (129, (3000,), 1600, 4, torch.float16),              # 4 of 7
    (257, (3000,), 1600, 4, torch.float16),              # 2 of 7
    (300, (2040, 1000, 20), 2240, 3, torch.float16),     # three matrices
    # rows_gemm_kernel, several column tiles a workgroup: the last workgroup's past the last
    # matrix, one matrix's tiles beside the next one's
    (3, (8201,), 512, 2, torch.float16),                 # 2 column tiles, 2 waves each
    (8, (16500,), 320, 2, torch.bfloat16),               # 4, two bf16 addends a value
    (20, (8000, 300, 17), 256, 3, torch.bfloat16),       # 2
    (64, (12300,), 64, 4, torch.float16),                # 3
    (100, (8200, 33), 128, 4, torch.float32),            # 4, two row blocks
    (200, (8201,), 64, 3, torch.float16),                # 8, four row blocks
])
def test_rows_gemm_plans(dev, M, rows, n, bpw, cb_dtype):
    seed = 9700 + M
    ms = [synth.vq_matrix(seed + i, r, n, bpw=bpw) for i, r in enumerate(rows)]
    cb0, cb1 = _books(seed + 10, bpw, cb_dtype)
    x = synth.activations(seed + 12, (M, n), dtype=torch.float32).to(dev)
    mats = [tuple(_on(dev, m["idx0"], m["idx1"], m["scale"])) + (r,) for m, r in zip(ms, rows)]
    ys = K.vq_rows_gemm(x, mats, *_on(dev, cb0, cb1), n, hb=0)
    xr = fp16_row_scaled(x.cpu().numpy())
    h0, h1 = cb0.half(), None if cb1 is None else cb1.half()
    for y, m in zip(ys, ms):
        ref = O.np_gemv64(xr, m["idx0"], m["idx1"], h0, h1, m["scale"])
        assert np.all(np.abs(y.cpu().numpy() - ref) <= TOL_SUM * np.abs(ref).max(1, keepdims=True))


def test_rows_gemm_unaligned_rows_row_scales_and_nan(dev):
    """Rows that start 2 bytes off a 16-byte line, rows of 1e6 and 1e-6 and of
    zeros, and a NaN that stays in its row."""
    M, rows, n = 21, 300, 1024
    m = synth.vq_matrix(9951, rows, n, bpw=2)
    cb0, _ = _books(9952, 2, torch.float16)
    x = synth.activations(9953, (M, n), dtype=torch.float32)
    x[3] *= 1e6
    x[4] *= 1e-6
    x[5] = 0
    buf = torch.zeros(M * n + 1, dtype=torch.bfloat16, device=dev)
    buf[1:] = x.to(torch.bfloat16).reshape(-1).to(dev)
    xb = buf[1:].view(M, n)
    mats = [tuple(_on(dev, m["idx0"], None, m["scale"])) + (rows,)]
    (y,) = K.vq_rows_gemm(xb, mats, cb0.to(dev), None, n, hb=0)
    _check(y, xb.float().cpu().numpy(), m, cb0, None)
    assert bool((y[5] == 0).all())
    xn = xb.clone()
    xn[7, 11] = float("nan")
    (yn,) = K.vq_rows_gemm(xn, mats, cb0.to(dev), None, n, hb=0)
    assert bool(torch.isnan(yn[7]).all())
    keep = [i for i in range(M) if i != 7]
    assert torch.equal(yn[keep], y[keep])


@pytest.mark.parametrize("cfg,n,outs,M", [((16,), 2048, (2048, 512, 500), 5), ((16,), 2048, (2040, 512, 500), 333), ((16, 16), 512, (96, 17, 1, 33), 100),
                                          ((16, 8), 6144, (512, 256), 9)])
def test_projections_of_many_rows_equal_their_own_calls(dev, cfg, n, outs, M):
    """One launch for all matrices of a PackedProjections gives each module's
    own result to the order of fp32 sums (the K split depends on the launch)."""
    cbs = {"16": synth.codebook(9960).to(dev), "16_8": synth.codebook(9961, rows=256).to(dev),
           "16_16": synth.codebook(9962).to(dev)}
    lins = []
    for i, out in enumerate(outs):
        m = synth.vq_matrix(9963 + i, out, n, bpw={1: 2, 2: 4}[len(cfg)] if 8 not in cfg else 3)
        lins.append(PackedLinear((out, n), cfg, "t", [p for p in (m["idx0"], m["idx1"]) if p is not None], m["scale"],
                                 cbs, dev))
    x = synth.activations(9970, (M, n), dtype=torch.float32).to(dev)
    proj = PackedProjections(lins)
    for y, lin in zip(proj(x), lins):
        ref = lin(x)
        assert y.shape == (M, lin.out)
        assert float((y - ref).abs().max()) <= TOL_SUM * float(ref.abs().max())


@pytest.mark.parametrize("cfg,n,outs", [((16,), 2048, (2048, 512, 500)), ((16, 8), 512, (300, 17)),
                                        ((16, 16), 6144, (500, 512)), ((16, 16), 128, (33,))])
@pytest.mark.parametrize("M", [3, 8])
def test_bf16_centroids_enter_as_they_are(dev, cfg, n, outs, M):
    """Up to 8 rows, bf16 codebooks whose values fp16 cannot hold (above
    65504, and below its smallest) count with all their bits, as in the sorted
    batch kernel, which takes projections of a few rows without planes."""
    big, tiny = 2.0 ** 30, 2.0 ** -30
    for scale in (big, tiny):
        cbs = {"16": (synth.codebook(9940).float() * scale).bfloat16(),
               "16_8": (synth.codebook(9941, rows=256).float() * scale).bfloat16(),
               "16_16": (synth.codebook(9942).float() * scale).bfloat16()}
        on = {k: v.to(dev) for k, v in cbs.items()}
        bpw = {(16,): 2, (16, 8): 3, (16, 16): 4}[cfg]
        ms = [synth.vq_matrix(9943 + i, out, n, bpw=bpw) for i, out in enumerate(outs)]
        lins = [PackedLinear((out, n), cfg, "t", [p for p in (m["idx0"], m["idx1"]) if p is not None], m["scale"], on,
                             dev) for m, out in zip(ms, outs)]
        x = synth.activations(9950, (M, n), dtype=torch.float32).to(dev)
        xr = lins[0].rot.fwd(x).cpu().numpy()
        cb1 = {2: None, 3: cbs["16_8"], 4: cbs["16_16"]}[bpw]
        for y, m, lin in zip(PackedProjections(lins)(x), ms, lins):
            _, ref = O.vq_gemv(fp16_row_scaled(xr), m["idx0"], m["idx1"], cbs["16"], cb1, lin.scale.cpu())
            err = np.abs(y.cpu().numpy() - ref).max(1)
            assert np.all(err <= TOL_SUM * np.abs(ref).max(1)), (scale, err.max() / np.abs(ref).max())


def test_rows_gemm_capture_replays_and_repeats(dev):
    """A captured call whose tiles are summed over workgroups gives the eager
    result bit for bit on every replay, with new inputs and eager calls
    between."""
    M, rows, n = 16, 512, 6144
    m = synth.vq_matrix(9981, rows, n, bpw=4)
    cb0, cb1 = _on(dev, *_books(9982, 4, torch.bfloat16))
    mats = [tuple(_on(dev, m["idx0"], m["idx1"], m["scale"])) + (rows,)]
    xs = [synth.activations(9983 + i, (M, n)).to(dev) for i in range(3)]
    static = xs[0].clone()
    K.vq_rows_gemm(static, mats, cb0, cb1, n)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        (out,) = K.vq_rows_gemm(static, mats, cb0, cb1, n)
    for i in range(6):
        static.copy_(xs[i % 3])
        g.replay()
        (ref,) = K.vq_rows_gemm(xs[i % 3], mats, cb0, cb1, n)
        torch.cuda.synchronize()
        assert torch.equal(out, ref), i


def test_rows_gemm_refuses(dev):
    m = synth.vq_matrix(9990, 16, 512, bpw=2)
    i0, sc, cb = _on(dev, m["idx0"], m["scale"], synth.codebook(9991))
    x = torch.zeros(4, 512, dtype=torch.float16, device=dev)
    with pytest.raises(Vq2Error, match="multiple of 64"):
        K.vq_rows_gemm(x[:, :72].contiguous(), [(i0[:, :9].contiguous(), None, sc, 16)], cb, None, 72)
    with pytest.raises(Vq2Error, match="hb"):
        K.vq_rows_gemm(x, [(i0, None, sc, 16)], cb, None, 512, hb=32)
    with pytest.raises(Vq2Error, match="perm"):
        K.vq_rows_gemm(x, [(i0, None, sc, 16)], cb, None, 512, perm=torch.zeros(8, dtype=torch.int32, device=dev))
    off = torch.zeros(16 * 64 + 4, dtype=torch.int16, device=dev)[4:].view(16, 64)
    with pytest.raises(Vq2Error, match="16-byte aligned"):
        K.vq_rows_gemm(x, [(off, None, sc, 16)], cb, None, 512, hb=512)

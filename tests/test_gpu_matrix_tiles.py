"""The matrix-core forms for fp32 activations and for many activation rows, at
the edges of their tiles: the direct form with one and two row tiles per wave,
the packed operand (up to eight rows) and one to three 16-row tiles; the tiled
form in each of its workgroup shapes, fp16 and fp32 activations. Partial tiles,
ranges of K with and without steps, rows whose last step or block is partial and
rows of more than one 64-chunk group, strided rows of x and y, one value far
above its block's others and a row of another magnitude beside it."""
import os

import numpy as np
import pytest

import oracle
from rqmv import synth

pytestmark = pytest.mark.gpu

THREADS = min(16, os.cpu_count() or 1)
FMTS = ["q8_0", "q4_0", "q4_k", "q6_k"]


def limit(cols):
    """Relative 2-norm of the rounding: the activations' split to 2^-22 of a
    value, the products exact, and a chain of cols / 32 scaled block sums, each
    a product and an addition rounded in fp32 (their errors independent:
    2 * 2^-24 * sqrt(blocks)), with a factor of two for blocks that cancel."""
    return 2.0 * (2.0 ** -22 + 2.0 * 2.0 ** -24 * np.sqrt(cols / 32) + 2.0 ** -23)


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


def activations(m, ldx, xdt, seed):
    x = synth.activations_f32(m * ldx, seed=seed).reshape(m, ldx)
    if xdt == "f16":
        xh = synth.fp16_bits(x)
        return xh, synth.fp16_to_f32(xh)
    x[:, 5] *= 3e4
    x[m - 1] *= 1e-5
    return x, x


def check(gpu, fmt, rows, cols, xdt, ms, pad):
    w = synth.weights(fmt, rows, cols, seed=rows + cols)
    W = gpu.Weight(fmt, rows, cols, w)
    dt = gpu.DTYPE_F16 if xdt == "f16" else gpu.DTYPE_F32
    for m in ms:
        ldx, ldy = cols + pad, rows + pad
        xh, x32 = activations(m, ldx, xdt, seed=m + cols)
        yb = gpu.DeviceBuffer(4 * m * ldy)
        yb.fill_zero()
        W.matvec(gpu.DeviceBuffer.from_array(xh), dt, m, ldx, yb, ldy)
        gpu.synchronize()
        y = yb.download(np.float32).reshape(m, ldy)
        ref = oracle.matvec_f64(fmt, w, rows, cols, x32[:, :cols], threads=THREADS)
        for i in (range(m) if xdt == "f32" else [slice(None)]):  # (each row has a magnitude of its own)
            assert rel(y[i, :rows] if xdt == "f32" else y[:, :rows], ref[i]) <= limit(cols), (fmt, rows, cols, m, i)
        assert (y[:, rows:] == 0).all(), (fmt, rows, cols, m)
    W.close()


def shapes(fmt):
    return [(83, 768), (300, 5376), (16, 256)] if fmt in ("q4_k", "q6_k") else [(83, 800), (300, 4160), (16, 96)]


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("shape", ["11", "12", "22", "15", "14"])
@pytest.mark.parametrize("xdt", ["f16", "f32"])
def test_tiled(gpu, fmt, shape, xdt, monkeypatch):
    monkeypatch.setenv("RQMV_TILE", shape)
    for n, (rows, cols) in enumerate(shapes(fmt)):
        check(gpu, fmt, rows, cols, xdt, (3, 16, 33, 129), 0 if n else 8)


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("rt,wk", [("1", "8"), ("2", "8"), ("2", "4"), ("2", "1")])
def test_direct_f32(gpu, fmt, rt, wk, monkeypatch):
    monkeypatch.setenv("RQMV_TILE", "0")
    monkeypatch.setenv("RQMV_DIRECT_RT", rt)
    monkeypatch.setenv("RQMV_DIRECT_WK", wk)
    for n, (rows, cols) in enumerate(shapes(fmt)):
        check(gpu, fmt, rows, cols, "f32", (5, 8, 9, 16, 17, 32, 33, 64, 77), 0 if n else 4)


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("xdt", ["f16", "f32"])
def test_as_planned(gpu, fmt, xdt):
    """The form and shape the plan takes, on both sides of its lines: few and many row
    tiles, short and long rows, 16-row groups that fall by ones, twos and threes."""
    short, longer = (512, 8448) if fmt in ("q4_k", "q6_k") else (480, 8416)
    for rows, cols in ((40, short), (4200, short), (40, longer)):
        check(gpu, fmt, rows, cols, xdt, (17, 33, 48, 65, 112, 145), 0)


@pytest.mark.parametrize("tile,rt", [("0", "1"), ("0", "2"), ("11", ""), ("22", ""), ("14", "")])
@pytest.mark.parametrize("big,scale", [(1e5, 0), (1e4, 1)])
def test_q6_k_f32_groups_of_unlike_scales(gpu, big, scale, tile, rt, monkeypatch):
    """fp32 activations, one value far above the others in a 16-weight group whose scale
    is 0 or 1, beside a group of scale about 100: the other group's sum keeps its bits.
    Each group is a product of its own, scaled on its own, so the limit is the one of
    ordinary activations (the large value's terms are as large as the whole sum)."""
    monkeypatch.setenv("RQMV_TILE", tile)
    monkeypatch.setenv("RQMV_DIRECT_RT", rt)
    rows, cols = 83, 768
    w = np.array(synth.weights("q6_k", rows, cols, seed=11)).reshape(-1, 210)
    w[:, 192:208] = np.random.default_rng(3).integers(90, 120, (len(w), 16))
    w[:: cols // 256, 192] = scale  # group 0 of every row
    w = w.reshape(-1)
    W = gpu.Weight("q6_k", rows, cols, w)
    for m in (5, 20, 70):
        x = synth.activations_f32(m * cols, seed=m).reshape(m, cols)
        x[:, 5] *= big
        yb = gpu.DeviceBuffer(4 * m * rows)
        W.matvec(gpu.DeviceBuffer.from_array(x), gpu.DTYPE_F32, m, cols, yb, rows)
        gpu.synchronize()
        y = yb.download(np.float32).reshape(m, rows)
        ref = oracle.matvec_f64("q6_k", w, rows, cols, x, threads=THREADS)
        assert rel(y, ref) <= limit(cols), (m, rel(y, ref))


@pytest.mark.parametrize("tile", ["11", "12", "15", "14"])
@pytest.mark.parametrize("scale", [-1, 1, -17])
def test_q6_k_f16_folded_scales(gpu, tile, scale, monkeypatch):
    """fp16 activations, every scale of the weight the same small number of either sign.
    Limit: a 256-weight block is eight accumulations (Q6_K's second product included,
    sixteen where the scale has both parts), each off by up to 2^-23 of a partial sum
    that grows with the square root of its length (sum of j / 8, j = 1..8: 4.5), and two
    fp32 roundings where the blocks are scaled and added."""
    monkeypatch.setenv("RQMV_TILE", tile)
    rows, cols = 83, 768
    w = np.array(synth.weights("q6_k", rows, cols, seed=12)).reshape(-1, 210)
    w[:, 192:208] = np.int8(scale).view(np.uint8)
    w = w.reshape(-1)
    W = gpu.Weight("q6_k", rows, cols, w)
    bound = 2.0 ** -23 * np.sqrt(4.5 if abs(scale) < 16 else 9.0) + 2.0 ** -23
    for m in (16, 70):
        xh, x = activations(m, cols, "f16", seed=m)
        yb = gpu.DeviceBuffer(4 * m * rows)
        W.matvec(gpu.DeviceBuffer.from_array(xh), gpu.DTYPE_F16, m, cols, yb, rows)
        gpu.synchronize()
        y = yb.download(np.float32).reshape(m, rows)
        ref = oracle.matvec_f64("q6_k", w, rows, cols, x, threads=THREADS)
        assert rel(y, ref) <= bound, (m, rel(y, ref), bound)


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("tile", ["0", "11", "14"])
def test_f32_activations_near_the_largest(gpu, fmt, tile, monkeypatch):
    """fp32 activations of up to 2e38, whose sum over a block overflows fp32, times
    weights small enough that no output does."""
    monkeypatch.setenv("RQMV_TILE", tile)
    rows, cols = 83, 768
    size, scales = {"q8_0": (34, [0]), "q4_0": (18, [0]), "q4_k": (144, [0, 2]), "q6_k": (210, [208])}[fmt]
    w = np.array(synth.weights(fmt, rows, cols, seed=13)).reshape(-1, size)
    for at in scales:
        d = np.ascontiguousarray(w[:, at:at + 2]).view(np.float16) * np.float16(2.0 ** -8)
        w[:, at:at + 2] = d.view(np.uint8)
    w = w.reshape(-1)
    W = gpu.Weight(fmt, rows, cols, w)
    for m in (5, 20, 70):
        x = (synth.activations_f32(m * cols, seed=m) * np.float32(5e37)).reshape(m, cols)
        x[:, :32] = np.abs(x[:, :32])
        yb = gpu.DeviceBuffer(4 * m * rows)
        W.matvec(gpu.DeviceBuffer.from_array(x), gpu.DTYPE_F32, m, cols, yb, rows)
        gpu.synchronize()
        y = yb.download(np.float32).reshape(m, rows)
        ref = oracle.matvec_f64(fmt, w, rows, cols, x, threads=THREADS)
        assert np.abs(ref).max() < 3e38 and np.isfinite(y).all(), (fmt, m)
        assert rel(y, ref) <= limit(cols), (fmt, m)


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("xdt", ["f16", "f32"])
@pytest.mark.parametrize("tile", ["0", "11", "22", "14"])
def test_non_finite_activations_stay_in_their_rows(gpu, fmt, xdt, tile, monkeypatch):
    """More than 32 rows, a NaN in one and an infinity in another: every output of those
    rows is non-finite, every other row keeps its bits."""
    monkeypatch.setenv("RQMV_TILE", tile)
    rows, cols, m = 83, 768, 70
    W = gpu.Weight(fmt, rows, cols, synth.weights(fmt, rows, cols, seed=14))
    dt = gpu.DTYPE_F16 if xdt == "f16" else gpu.DTYPE_F32
    x, _ = activations(m, cols, xdt, seed=15)
    out = []
    for bad in (False, True):
        if bad:
            x = x.copy()
            nan, inf = (0x7E00, 0x7C00) if xdt == "f16" else (np.nan, np.inf)
            x[3, 300], x[40, 511] = nan, inf
        yb = gpu.DeviceBuffer(4 * m * rows)
        W.matvec(gpu.DeviceBuffer.from_array(x), dt, m, cols, yb, rows)
        gpu.synchronize()
        out.append(yb.download(np.float32).reshape(m, rows))
    keep = np.ones(m, bool)
    keep[[3, 40]] = False
    assert np.isfinite(out[0]).all()
    assert not np.isfinite(out[1][~keep]).any()
    assert np.array_equal(out[0][keep].view(np.uint32), out[1][keep].view(np.uint32))


@pytest.mark.parametrize("fmt", ["q4_k", "q8_0"])
@pytest.mark.parametrize("xdt,tile", [("f32", "0"), ("f32", "11"), ("f16", "11")])
def test_activations_beyond_one_launch(gpu, fmt, xdt, tile, monkeypatch):
    """Activation rows so far apart that a launch's 32-bit offsets (4 GiB) reach only some
    of them: the rest go in further launches."""
    monkeypatch.setenv("RQMV_TILE", tile)
    rows, cols, m = 40, 512, 45
    size = 4 if xdt == "f32" else 2
    ldx = 108_000_000 // size  # 40 rows to 4 GiB
    w = synth.weights(fmt, rows, cols, seed=16)
    W = gpu.Weight(fmt, rows, cols, w)
    xh, x = activations(m, cols, xdt, seed=17)
    big, y = gpu.DeviceBuffer(((m - 1) * ldx + cols) * size), gpu.DeviceBuffer(4 * m * rows)
    for i in range(m):
        row = gpu.DeviceBuffer.from_array(xh[i])
        gpu.DeviceBuffer.copy_from(big.view(i * ldx * size, cols * size), row, cols * size)
        gpu.synchronize()
    W.matvec(big, gpu.DTYPE_F16 if xdt == "f16" else gpu.DTYPE_F32, m, ldx, y, rows)
    gpu.synchronize()
    ref = oracle.matvec_f64(fmt, w, rows, cols, x, threads=THREADS)
    got = y.download(np.float32).reshape(m, rows)
    for i in range(m):
        assert rel(got[i], ref[i]) <= limit(cols), (i, rel(got[i], ref[i]))


def test_f16_weights_beyond_one_launch(gpu):
    """More groups of sixteen rows than a launch's y dimension holds (65,535), and a rest:
    rows with equal activations have equal bits wherever they stand."""
    rows, cols, base, m = 3, 64, 4096, 16 * 65535 + 37
    w = synth.f16_weights(rows, cols, 0.05, seed=18)
    W = gpu.Weight("f16", rows, cols, w)
    xh = synth.activations_f16(base * cols, seed=19).reshape(base, cols)
    x = np.concatenate([xh] * (m // base + 1))[:m]
    y = gpu.DeviceBuffer(4 * m * rows)
    W.matvec(gpu.DeviceBuffer.from_array(x), gpu.DTYPE_F16, m, cols, y, rows)
    gpu.synchronize()
    got = y.download(np.float32).reshape(m, rows)
    ref = synth.fp16_to_f32(xh).astype(np.float64) @ synth.fp16_to_f32(w.view(np.uint16).reshape(rows, cols)).astype(np.float64).T
    assert rel(got[:base], ref) <= limit(cols)
    same = got.view(np.uint32) == np.concatenate([got[:base]] * (m // base + 1))[:m].view(np.uint32)
    assert same[: m - m % 16].all()  # whole groups of sixteen; the rest runs in smaller launches
    last = m - m % 16
    assert rel(got[last:], np.concatenate([ref] * (m // base + 1))[last:m]) <= limit(cols)

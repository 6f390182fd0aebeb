"""gguf_moe over batches: every position of a batch carries the bits of its own
one-position call, in every kernel form that batches take (the router's groups
of sixteen positions, the down product's blocks of rows with its encoded slot
activations, the gate/up product by blocks of the hidden width), over formats, widths that leave partial
row blocks and chunk rounds, a shared expert gated, ungated or absent, skewed
routing, and activations with outliers."""
import numpy as np
import pytest

from rqmv import synth

pytestmark = pytest.mark.gpu

# fmt, d_model, hidden, shared hidden, experts, top, gated
CASES = [("q4_k", 512, 256, 256, 16, 8, True), ("q4_k", 1280, 512, 0, 64, 6, False),
         ("q6_k", 768, 768, 256, 8, 2, False), ("q8_0", 576, 96, 160, 12, 4, True), ("q8_0", 1024, 512, 0, 60, 4, False),
         ("q4_0", 320, 64, 64, 5, 1, True), ("q4_0", 2048, 192, 320, 33, 8, True)]


def _moe(gpu, case, seed, scoring=0):
    fmt, d, h, hs, e, top, gated = case
    w = lambda rows, cols, tag, n=None: gpu.Weight(fmt, rows, cols, synth.weights(fmt, rows * (n or 1), cols, seed, tag),  # noqa: E731
                                                   **({} if n is None else {"experts": n}))
    shared = {}
    if hs:
        shared = dict(gate_sh=w(hs, d, "gs"), up_sh=w(hs, d, "us"), down_sh=w(d, hs, "ds"))
        if gated:
            shared["shared_gate_inp"] = gpu.Weight("f16", 1, d, synth.f16_weights(1, d, 0.02, seed, "sg"))
    return gpu.Moe(gpu.Weight("f16", e, d, synth.f16_weights(e, d, 0.05, seed, "r")), w(h, d, "g", e), w(h, d, "u", e),
                   w(d, h, "dn", e), top, scoring=scoring, **shared)


def _activations(m, d, xdt, kind, seed):
    x = synth.activations_f32(m * d, seed=seed).reshape(m, d)
    if kind == "skewed":  # most positions choose the same experts
        x[: 3 * m // 4] = x[0] + 0.01 * x[: 3 * m // 4]
    if kind == "outliers":
        x[::3, 7] *= 500.0
        x[1::3, 40:43] *= 100.0
    return synth.fp16_bits(x) if xdt == "f16" else x


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
@pytest.mark.parametrize("xdt,kind,m", [("f16", "plain", 17), ("f32", "outliers", 40), ("f16", "skewed", 70)])
def test_batches_carry_the_bits_of_single_positions(gpu, case, xdt, kind, m):
    d, e = case[1], case[4]
    moe = _moe(gpu, case, seed=sum(case[1:6]))
    x = _activations(m, d, xdt, kind, seed=m + d)
    xb, dt = gpu.DeviceBuffer.from_array(x), gpu.DTYPE_F16 if xdt == "f16" else gpu.DTYPE_F32
    ldy = d + 12
    y, route = gpu.DeviceBuffer(4 * m * ldy), gpu.DeviceBuffer(4 * m * e)
    y.fill_zero()
    for _ in range(2):  # (the second call finds the workspace as the first left it)
        moe.run_batch(xb, dt, m, d, y, ldy, route, moe.batch_workspace(m))
    gpu.synchronize()
    got, routes = y.download(np.float32).reshape(m, ldy), route.download(np.float32).reshape(m, e)
    assert np.isfinite(got).all()
    for p in range(m):
        y1, r1 = moe(x[p])
        assert np.array_equal(got[p, :d].view(np.uint32), y1.view(np.uint32)), (case, p)
        assert np.array_equal(routes[p].view(np.uint32), r1.view(np.uint32)), (case, p)
    assert (got[:, d:] == 0).all()


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
@pytest.mark.parametrize("blocks", ["0", "5", "16"])
def test_gate_up_by_blocks_of_rows(gpu, case, blocks, monkeypatch):
    """The gate/up product striding over a position's rows and by blocks of the hidden
    width: blocks that divide it, and blocks that leave partial and empty ones."""
    monkeypatch.setenv("RQMV_MOE_GLU_BLOCKS", blocks)
    d, m = case[1], 18
    moe = _moe(gpu, case, seed=sum(case[1:6]))
    x = _activations(m, d, "f32", "outliers", seed=m + d)
    y, route = gpu.DeviceBuffer(4 * m * d), gpu.DeviceBuffer(4 * m * case[4])
    y.fill_zero()
    moe.run_batch(gpu.DeviceBuffer.from_array(x), gpu.DTYPE_F32, m, d, y, d, route, moe.batch_workspace(m))
    gpu.synchronize()
    got, routes = y.download(np.float32).reshape(m, d), route.download(np.float32).reshape(m, case[4])
    for p in range(m):
        y1, r1 = moe(x[p])
        assert np.array_equal(got[p].view(np.uint32), y1.view(np.uint32)), (case, p)
        assert np.array_equal(routes[p].view(np.uint32), r1.view(np.uint32)), (case, p)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
@pytest.mark.parametrize("form", ["0", "1"])
def test_down_by_blocks_of_rows(gpu, case, form, monkeypatch):
    """The down product over whole positions and by blocks of output rows (64 rows, and
    128 from 48 positions), at sizes that the plan leaves to one of the two."""
    monkeypatch.setenv("RQMV_MOE_DOWN_BATCH", form)
    d = case[1]
    moe = _moe(gpu, case, seed=sum(case[1:6]))
    for m in (17, 50):
        x = _activations(m, d, "f32", "outliers", seed=m + d)
        y = gpu.DeviceBuffer(4 * m * d)
        y.fill_zero()
        moe.run_batch(gpu.DeviceBuffer.from_array(x), gpu.DTYPE_F32, m, d, y, d, None, moe.batch_workspace(m))
        gpu.synchronize()
        got = y.download(np.float32).reshape(m, d)
        for p in range(m):
            assert np.array_equal(got[p].view(np.uint32), moe(x[p])[0].view(np.uint32)), (case, p)

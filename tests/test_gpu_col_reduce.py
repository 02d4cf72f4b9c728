"""Column reductions (vdsl_op_col_reduce) at the sizes where its strips and row ranges can go wrong.

Sums are f64 sums rounded once, in another order than the oracle's: |gpu - oracle| <= one f32 ulp of
the result (both are within half an ulp of the same f64 value, whose own error, 16384 * 2^-53 *
sum|x|, is added).  Maxima are exact."""
import numpy as np
import pytest

from oracle import oracle
from vernondsl_amd import kernels, rng
from vernondsl_amd._lib import call
from vernondsl_amd.rhi import Queue, Tensor

pytestmark = pytest.mark.gpu

# one row; fewer rows than row lanes; a partial batch; a last row range of one row (4097 over 256-row
# ranges); strips past the last column; odd, even and 16-byte widths; enough bytes for several ranges
SHAPES = [(1, 1), (1, 5), (3, 64), (63, 260), (1000, 333), (4097, 256), (4097, 72), (16384, 3), (8193, 130), (2049, 1031),
          (300, 16384), (5, 40000), (64, 32768), (8, 1 << 20), (33, 65544),
          # few rows: a lane per column or vector, small and wide, ragged; the widest strips of 1024 lanes
          (12, 333), (16, 70001), (17, 70001), (7, 600008), (2, 1100002), (9, 300000), (65, 131080)]


def check(xf, cs, cm):
    x64 = xf.astype(np.float64)
    ref = x64.sum(axis=0)
    bound = np.spacing(np.abs(ref).astype(np.float32)).astype(np.float64) + 16384 * 2.0 ** -53 * np.abs(x64).sum(axis=0)
    assert np.all(np.abs(cs.astype(np.float64) - ref) <= bound)
    assert np.array_equal(cm, xf.max(axis=0))


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_shapes(dev, q, rows, cols, bf16):
    x = rng.normal(rows * 131 + cols, rows * cols, 0.0, 2.0).reshape(rows, cols)
    xh = rng.f32_to_bf16(x) if bf16 else x
    tx = Tensor.from_numpy(dev, q, xh, "bf16" if bf16 else "f32")
    out = [Tensor(dev, (cols,), "f32") for _ in range(4)]
    for t in out:
        t.buffer.fill_u32(q, 0x7FC00000)
    kernels.col_reduce(q, tx, out[0], out[1])
    kernels.col_reduce(q, tx, out[2], None)  # each output alone
    kernels.col_reduce(q, tx, None, out[3])
    xf = rng.bf16_to_f32(xh) if bf16 else xh
    check(xf, out[0].numpy(q), out[1].numpy(q))
    assert np.array_equal(out[0].numpy(q), out[2].numpy(q)) and np.array_equal(out[1].numpy(q), out[3].numpy(q))
    for t in [tx] + out:
        t.free()


def test_special_values(dev, q):
    """Infinities and NaN in their columns only; a column of -inf keeps its maximum; no rows at all."""
    x = rng.normal(9, 6000 * 100).reshape(6000, 100)
    x[17, 3], x[5999, 4], x[4000, 5], x[:, 6] = np.inf, -np.inf, np.nan, -np.inf
    tx = Tensor.from_numpy(dev, q, x)
    cs, cm = Tensor(dev, (100,), "f32"), Tensor(dev, (100,), "f32")
    kernels.col_reduce(q, tx, cs, cm)
    rs, rm = oracle.col_reduce(x)
    s, m = cs.numpy(q), cm.numpy(q)
    assert np.array_equal(m, rm) and np.array_equal(np.isnan(s), np.isnan(rs))
    assert s[3] == np.inf and s[4] == -np.inf and np.isnan(s[5]) and m[6] == -np.inf
    empty = Tensor(dev, (0, 100), "f32")
    kernels.col_reduce(q, empty, cs, cm)
    assert np.all(cs.numpy(q) == 0.0) and np.all(cm.numpy(q) == -np.inf)
    for t in (tx, cs, cm, empty):
        t.free()


def test_recorded_and_on_two_queues(dev, q):
    """Two reductions in one recorded graph and eager calls on two queues between its replays: the
    partial results of each stay apart."""
    xs = [rng.normal(k, 9000 * 512).reshape(9000, 512) for k in range(3)]
    tx = [Tensor.from_numpy(dev, q, x) for x in xs]
    out = [(Tensor(dev, (512,), "f32"), Tensor(dev, (512,), "f32")) for _ in xs]
    ref = []
    for t, o in zip(tx, out):
        kernels.col_reduce(q, t, *o)
        ref.append((o[0].numpy(q), o[1].numpy(q)))
    other = Queue(dev)
    with q.capture() as rec:
        kernels.col_reduce(q, tx[0], *out[0])
        kernels.col_reduce(q, tx[1], *out[1])
    for _ in range(4):
        for o in out:
            o[0].buffer.fill_u32(q, 0x7FC00000)
        q.sync()
        rec.graph.launch(q)
        kernels.col_reduce(other, tx[2], *out[2])
        q.sync()
        other.sync()
        for o, r in zip(out, ref):
            assert np.array_equal(o[0].numpy(q), r[0]) and np.array_equal(o[1].numpy(q), r[1])
        kernels.col_reduce(q, tx[1], *out[1])  # the queue's own scratch, between replays
        assert np.array_equal(out[1][0].numpy(q), ref[1][0])
    rec.graph.destroy()
    other.destroy()
    for t in tx + [t for o in out for t in o]:
        t.free()


def test_while_another_queue_records(dev):
    """A queue made, its first reduction, and a graph with scratch freed while another queue of the thread
    records: all succeed, the recording too, with the results of the same calls alone."""
    x = rng.normal(3, 9000 * 512).reshape(9000, 512)
    a = Queue(dev)
    tx = Tensor.from_numpy(dev, a, x)
    out = [(Tensor(dev, (512,), "f32"), Tensor(dev, (512,), "f32")) for _ in range(2)]
    kernels.col_reduce(a, tx, *out[0])
    ref = out[0][0].numpy(a), out[0][1].numpy(a)
    with a.capture() as old:
        kernels.col_reduce(a, tx, *out[1])
    with a.capture() as rec:
        b = Queue(dev)
        kernels.col_reduce(b, tx, *out[1])
        kernels.col_reduce(a, tx, *out[0])
        old.graph.destroy()
    assert np.array_equal(out[1][0].numpy(b), ref[0]) and np.array_equal(out[1][1].numpy(b), ref[1])
    for _ in range(3):
        for t in out[0]:
            t.buffer.fill_u32(a, 0x7FC00000)
        rec.graph.launch(a)
        assert np.array_equal(out[0][0].numpy(a), ref[0]) and np.array_equal(out[0][1].numpy(a), ref[1])
    rec.graph.destroy()
    b.destroy()
    a.destroy()
    for t in [tx] + [t for o in out for t in o]:
        t.free()


@pytest.mark.parametrize("shape", [(9000, 512), (20000, 77)])
def test_without_scratch(dev, q, shape):
    """A queue and a recording that get no scratch memory: one range of rows, right all the same."""
    x = rng.normal(5, shape[0] * shape[1]).reshape(shape)
    out = [Tensor(dev, (shape[1],), "f32") for _ in range(4)]
    tx = Tensor.from_numpy(dev, q, x)
    call("vdsl_debug_fail_alloc_after", 0)
    try:
        a = Queue(dev)
        with a.capture() as rec:
            kernels.col_reduce(a, tx, *out[2:])
    finally:
        call("vdsl_debug_fail_alloc_after", -1)
    kernels.col_reduce(a, tx, *out[:2])
    for _ in range(2):
        for t in out[2:]:
            t.buffer.fill_u32(a, 0x7FC00000)
        rec.graph.launch(a)
        a.sync()
    check(x, out[0].numpy(a), out[1].numpy(a))
    for t, u in zip(out[:2], out[2:]):
        assert np.array_equal(t.numpy(a), u.numpy(a))
    rec.graph.destroy()
    a.destroy()
    for t in [tx] + out:
        t.free()

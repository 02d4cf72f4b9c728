"""Reductions over a grid (histograms, sums) whose blocks go through bands of 8 or 16 rows, on grids of
one band, of a band and one row, of ragged columns, and of several bands a block.  int32 targets are
exact in any order; f32 targets of small dyadic values too (every partial sum is a multiple of 2^-4
below 2^20)."""
import numpy as np
import pytest

from vernondsl_amd import kernels, pixprog as pp
from vernondsl_amd.rhi import Tensor

pytestmark = pytest.mark.gpu


def program(bins, n, dtype, store):
    """target k < n: [0][floor(x * bins) + k] += k + 1 (an add past the last bin is dropped); the last
    target: a sum of x at a constant index; with store, out = x."""
    b = pp.Builder()
    x = b.load(0)
    at = b.op("floor", b.op("mul", x, float(bins)))
    fx = [b.scatter_add(1 + k, 0.0, b.op("add", at, float(k)) if k else at, float(k + 1)) for k in range(n)]
    fx.append(b.scatter_add(1 + n, 0.0, 0.0, x))
    return pp.compile_program(b, out=x if store else None, effects=fx, in_dtypes=[pp.F32] + [dtype] * n + [pp.F32],
                              in_extents=[None] + [(1, bins)] * n + [(1, 1)])


@pytest.mark.parametrize("store", [False, True])
@pytest.mark.parametrize("n, dtype", [(1, pp.I32), (2, pp.I32), (3, pp.I32), (1, pp.F32), (5, pp.I32)])
@pytest.mark.parametrize("ni, nj", [(1, 1), (15, 255), (16, 256), (17, 257), (33, 64), (64, 1000), (1500, 1027)])
def test_bands(dev, q, ni, nj, n, dtype, store):
    bins = 100
    x = (np.random.default_rng(ni + nj + n).integers(-2, 18, (ni, nj)) / 16.0).astype(np.float32)  # some outside [0, 1)
    at = np.floor(x.astype(np.float64) * bins).astype(int)
    tx, out = Tensor.from_numpy(dev, q, x), Tensor(dev, (ni, nj), "f32") if store else None
    ts = [Tensor.from_numpy(dev, q, np.full((1, bins), k, np.int32 if dtype == pp.I32 else np.float32)) for k in range(n)]
    total = Tensor.from_numpy(dev, q, np.zeros((1, 1), np.float32))
    kernels.pixel_program(q, program(bins, n, dtype, store), [tx] + ts + [total], out, grid=(ni, nj))
    for k, t in enumerate(ts):
        e = (at + k)[(at + k >= 0) & (at + k < bins)]
        want = k + (k + 1) * np.bincount(e, minlength=bins)
        assert np.array_equal(t.numpy(q).astype(np.int64)[0], want)
    assert np.abs(x).sum(dtype=np.float64) < 2 ** 20  # multiples of 2^-4 below 2^20: 24 bits, every sum exact
    assert total.numpy(q)[0, 0] == x.sum(dtype=np.float64)
    if store:
        assert np.array_equal(out.numpy(q), x)
    for t in [tx, total] + ts + ([out] if store else []):
        t.free()


def int_program(bins, n, total, per_row):
    """target k < n: [0][floor(x * bins) + k] += k + 1, or with per_row [0][floor(i / 128)] += 1; with total,
    an int32 sum of 16 x at a constant index."""
    b = pp.Builder()
    x = b.load(0)
    at = b.op("floor", b.op("mul", b.index(0), 1.0 / 128)) if per_row else b.op("floor", b.op("mul", x, float(bins)))
    fx = [b.scatter_add(1 + k, 0.0, b.op("add", at, float(k)) if k else at, float(k + 1)) for k in range(n)]
    if total:
        fx.append(b.scatter_add(1 + n, 0.0, 0.0, b.op("mul", x, 16.0)))
    return pp.compile_program(b, effects=fx, in_dtypes=[pp.F32] + [pp.I32] * (n + total),
                              in_extents=[None] + [(1, bins)] * n + [(1, 1)] * total)


# int32 targets alone: the root rule gives 2 to 3 bands a block on the first four grids (the last block's of
# fewer rows, or of fewer bands), adds at row-uniform indices several once 4096 units of a band are passed
@pytest.mark.parametrize("ni, nj, n, total, per_row", [(1500, 1027, 1, 0, False), (1505, 1027, 2, 1, False), (1501, 1027, 3, 1, False),
                                                       (4099, 700, 0, 1, False), (8203, 2050, 1, 0, True), (8203, 2050, 1, 1, True)])
def test_int32_bands(dev, q, ni, nj, n, total, per_row):
    bins = 100
    x = (np.random.default_rng(ni + n).integers(-2, 18, (ni, nj)) / 16.0).astype(np.float32)
    tx = Tensor.from_numpy(dev, q, x)
    ts = [Tensor.from_numpy(dev, q, np.full((1, bins), k, np.int32)) for k in range(n)]
    sums = [Tensor.from_numpy(dev, q, np.zeros((1, 1), np.int32))] if total else []
    kernels.pixel_program(q, int_program(bins, n, total, per_row), [tx] + ts + sums, None, grid=(ni, nj))
    at = np.repeat(np.arange(ni) // 128, nj) if per_row else np.floor(x.astype(np.float64) * bins).astype(int)
    for k, t in enumerate(ts):
        e = (at + k)[(at + k >= 0) & (at + k < bins)]
        assert np.array_equal(t.numpy(q).astype(np.int64)[0], k + (k + 1) * np.bincount(e, minlength=bins))
    for t in sums:
        assert t.numpy(q)[0, 0] == int((x.astype(np.float64) * 16).sum())
    for t in [tx] + ts + sums:
        t.free()


# grids of more bands of 8 rows than a launch's y extent (65535), up to the most rows a program may have;
# f32 totals (64 rows a block) and int32 ones
@pytest.mark.parametrize("ni, nj", [(524281, 1), (600000, 3), (1048560, 1)])
@pytest.mark.parametrize("f32", [True, False])
def test_tall(dev, q, ni, nj, f32):
    bins, n = 100, 3
    r = np.random.default_rng(ni)
    x = (r.integers(-2, 18, (ni, nj)) / 16.0 * (r.random((ni, nj)) < 0.25)).astype(np.float32)
    at = np.floor(x.astype(np.float64) * bins).astype(int)
    tx, total = Tensor.from_numpy(dev, q, x), Tensor.from_numpy(dev, q, np.zeros((1, 1), np.float32 if f32 else np.int32))
    ts = [Tensor.from_numpy(dev, q, np.full((1, bins), k, np.int32)) for k in range(n)]
    prog = program(bins, n, pp.I32, False) if f32 else int_program(bins, n, 1, False)
    kernels.pixel_program(q, prog, [tx] + ts + [total], None, grid=(ni, nj))
    for k, t in enumerate(ts):
        e = (at + k)[(at + k >= 0) & (at + k < bins)]
        assert np.array_equal(t.numpy(q).astype(np.int64)[0], k + (k + 1) * np.bincount(e, minlength=bins))
    assert np.abs(x).sum(dtype=np.float64) < 2 ** 20
    assert total.numpy(q)[0, 0] == x.sum(dtype=np.float64) * (1 if f32 else 16)
    for t in [tx, total] + ts:
        t.free()

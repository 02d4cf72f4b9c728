"""Row reductions + softmax at widths that take the masked register-resident kernel
(row_softmax_any): rows that start anywhere in a 16-byte vector, groups of 1 to 64 lanes per row, one
and several waves per row, the widest row it holds and the streaming kernel just past it.

Row sums are f64 sums rounded once (one f32 ulp from the oracle's, plus the f64 error), maxima exact,
f32 softmax within 1e-6 + 2^-24 |x - max| relative: the difference n = x - max is rounded to f32, an
absolute error of at most 2^-24 |n| that exp turns into a relative one; then exp 2e-7 + 1 ulp, the
sum and the quotient 1 ulp each; subnormal results are multiples of 2^-149, so 1e-44 absolute.  bf16:
the same, rounded: one bf16 ulp."""
import numpy as np
import pytest

from vernondsl_amd import kernels, rng
from vernondsl_amd.rhi import Tensor

pytestmark = pytest.mark.gpu

WIDTHS = [1, 3, 4, 5, 9, 31, 33, 63, 65, 127, 255, 257, 1021, 1027, 1031, 2051, 5003, 6149, 8191, 12001, 16383, 32764, 32771]


def run(dev, q, xh, dtype, pad=64):
    rows, cols = xh.shape
    x = Tensor.from_numpy(dev, q, xh, dtype)
    s, m, sm = Tensor(dev, (rows,), "f32"), Tensor(dev, (rows,), "f32"), Tensor(dev, (rows * cols + pad,), dtype)
    sm.buffer.fill_u32(q, 0x7FC17FC1, nbytes=sm.buffer.nbytes // 4 * 4)
    before = sm.numpy(q)
    kernels.row_reduce_softmax(q, x, s, m, _front(sm, rows, cols))
    got = sm.numpy(q)
    assert np.array_equal(got[rows * cols:].view(np.uint8), before[rows * cols:].view(np.uint8))  # nothing past the end
    res = s.numpy(q), m.numpy(q), got[:rows * cols].reshape(rows, cols)
    for t in (x, s, m, sm):
        t.free()
    return res


def _front(t, rows, cols):
    v = t.view(t.shape)
    v.shape, v.numel = (rows, cols), rows * cols
    return v


@pytest.mark.parametrize("bf16", [False, True])
# 17 to 256 columns run the streaming kernel up to 2000 rows
@pytest.mark.parametrize("cols, rows", [(c, 7 if c > 300 else 261) for c in WIDTHS] + [(c, 2001) for c in WIDTHS if 16 < c <= 300])
def test_widths(dev, q, cols, rows, bf16):
    x = rng.normal(cols, rows * cols, 0.0, 2.0).reshape(rows, cols)
    x[rows // 2, cols // 2] += np.float32(20.0)
    x[0, 0] -= np.float32(100.0)  # a subnormal share where the row has other elements
    xh = rng.f32_to_bf16(x) if bf16 else x
    xf = rng.bf16_to_f32(xh) if bf16 else xh
    gs, gm, gsm = run(dev, q, xh, "bf16" if bf16 else "f32")
    x64 = xf.astype(np.float64)
    ref = x64.sum(axis=1)
    bound = np.spacing(np.abs(ref).astype(np.float32)).astype(np.float64) + cols * 2.0 ** -53 * np.abs(x64).sum(axis=1)
    assert np.all(np.abs(gs.astype(np.float64) - ref) <= bound)
    assert np.array_equal(gm, xf.max(axis=1))
    n = x64 - x64.max(axis=1, keepdims=True)
    e = np.exp(n)
    p = e / e.sum(axis=1, keepdims=True)
    if bf16:
        assert np.all(np.abs(rng.bf16_to_f32(gsm).astype(np.float64) - p) <= 2.0 ** -7 * p + 1e-40)
    else:
        assert np.all(np.abs(gsm.astype(np.float64) - p) <= (1e-6 + 2.0 ** -24 * np.abs(n)) * p + 1e-44)


@pytest.mark.parametrize("cols", [5, 70, 300, 1001, 5003])
def test_special_values(dev, q, cols):
    """Rows with NaN, +inf or only -inf are NaN throughout, as x - max gives; -inf elements are 0; the
    neighbouring rows, whose ends share a vector with them, are not touched."""
    x = rng.normal(cols + 1, 9 * cols).reshape(9, cols)
    x[1, cols - 1], x[3, 0], x[5, :], x[7, 0], x[7, cols - 1] = np.nan, np.inf, -np.inf, -np.inf, -np.inf
    gs, gm, gsm = run(dev, q, x, "f32")
    for r in (1, 3, 5):
        assert np.all(np.isnan(gsm[r]))
    assert np.isnan(gs[1]) and gs[3] == np.inf and gs[5] == -np.inf and gm[3] == np.inf and gm[5] == -np.inf
    assert gm[1] == np.nanmax(x[1])
    for r in (0, 2, 4, 6, 7, 8):
        e = np.exp(x[r].astype(np.float64) - x[r].max())
        assert np.all(np.abs(gsm[r] - e / e.sum()) <= 2e-6 * (e / e.sum()))  # |x - max| <= 16
    assert gsm[7, 0] == 0.0 and gsm[7, cols - 1] == 0.0


def test_in_place(dev, q):
    """softmax may be x itself: a row is read before any of it is written."""
    x = rng.normal(5, 500 * 1003).reshape(500, 1003)
    t, out = Tensor.from_numpy(dev, q, x), Tensor(dev, (500, 1003), "f32")
    kernels.row_reduce_softmax(q, t, softmax=out)
    kernels.row_reduce_softmax(q, t, softmax=t)
    assert np.array_equal(t.numpy(q), out.numpy(q))
    t.free()
    out.free()

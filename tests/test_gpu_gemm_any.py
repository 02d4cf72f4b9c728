"""bf16 products read as they are stored (gemm_any.h): all four layouts, extents that end inside a tile,
inside a 16-byte load and inside a K stage, operands of fewer rows than a load has elements, both tile
sizes, the GELU-backward epilogue.

Results against f64 within K 2^-24 sum|a||b| (f32 sums in some order); all layouts of one product and,
where a tile configuration can run it, that configuration, bit for bit."""
import numpy as np
import pytest

from vernondsl_amd import _lib, kernels, rng
from vernondsl_amd._lib import call
from vernondsl_amd.rhi import Tensor

pytestmark = pytest.mark.gpu

# transposed layouts with short sides run here too (1 .. 9 rows: a 16-byte load spans rows); 64 x 64 and
# 128 x 128 tiles (2000 x 2100); K of one value, one stage, a stage and a part
SHAPES = [(1, 8, 1), (3, 1, 9), (5, 7, 64), (8, 9, 65), (1, 70, 130), (65, 1, 71), (63, 129, 72), (130, 140, 13), (200, 131, 300),
          (129, 257, 1001), (128, 192, 128), (2000, 2100, 45), (1999, 2101, 100)]


def product(dev, q, a, b, ta, tb, M, N, K, epi=_lib.EPI_NONE):
    A, B = np.ascontiguousarray(a.T) if ta else a, b if tb else np.ascontiguousarray(b.T)
    t = [Tensor.from_numpy(dev, q, A, "bf16"), Tensor.from_numpy(dev, q, B, "bf16"), Tensor(dev, (M, N), "f32"),
         Tensor(dev, (max(1, kernels.gemm_bf16_workspace_bytes(ta, tb, M, N, K)),), "i8")]
    t[2].buffer.fill_u32(q, 0x7FC00000)
    kernels.gemm_bf16(q, t[0], t[1], t[2], bool(ta), bool(tb), epi, None, t[3])
    out = t[2].numpy(q)
    for v in t:
        v.free()
    return out


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_layouts(dev, q, M, N, K):
    a = rng.f32_to_bf16(rng.uniform(M + K, M * K, -1, 1)).reshape(M, K)
    b = rng.f32_to_bf16(rng.uniform(N + K + 1, N * K, -1, 1)).reshape(N, K)
    af, bf = rng.bf16_to_f32(a).astype(np.float64), rng.bf16_to_f32(b).astype(np.float64)
    ref, bound = af @ bf.T, K * 2.0 ** -24 * (np.abs(af) @ np.abs(bf).T)
    got = {(ta, tb): product(dev, q, a, b, ta, tb, M, N, K) for ta in (0, 1) for tb in (0, 1)}
    for g in got.values():
        assert np.all(np.abs(g - ref) <= bound)
    assert all(np.array_equal(got[0, 0], g) for g in got.values())
    if K % 8 == 0:
        call("vdsl_debug_gemm_config", 0)
        try:
            assert np.array_equal(product(dev, q, a, b, 0, 1, M, N, K), got[0, 0])
        finally:
            call("vdsl_debug_gemm_config", -1)


def test_nan_past_the_ends(dev, q):
    """Values read past a row's, a column's or K's end reach no stored element: NaN in the first and last
    K value of one row of either operand marks that row's outputs only."""
    M, N, K = 131, 75, 69
    a = rng.f32_to_bf16(rng.uniform(1, M * K, -1, 1)).reshape(M, K)
    b = rng.f32_to_bf16(rng.uniform(2, N * K, -1, 1)).reshape(N, K)
    a[130, 0] = b[0, K - 1] = 0x7FC0
    want = np.zeros((M, N), bool)
    want[130, :] = want[:, 0] = True
    for ta, tb in ((0, 0), (1, 0), (1, 1)):
        assert np.array_equal(np.isnan(product(dev, q, a, b, ta, tb, M, N, K)), want), (ta, tb)


@pytest.mark.parametrize("M,N,K", [(300, 200, 100), (137, 131, 13)])
def test_epilogues(dev, q, M, N, K):
    a = rng.f32_to_bf16(rng.uniform(5, M * K, -1, 1)).reshape(M, K)
    b = rng.f32_to_bf16(rng.uniform(6, N * K, -1, 1)).reshape(N, K)
    plain = product(dev, q, a, b, 0, 1, M, N, K)
    assert np.array_equal(product(dev, q, a, b, 1, 0, M, N, K, _lib.EPI_RELU), np.maximum(plain, 0))
    ta, tb, pre, da, da_t = (Tensor.from_numpy(dev, q, a, "bf16"), Tensor.from_numpy(dev, q, b, "bf16"),
                             Tensor.from_numpy(dev, q, plain), Tensor(dev, (M, N), "bf16"), Tensor(dev, (N, M), "bf16"))
    ref, ref_t = Tensor(dev, (M, N), "bf16"), Tensor(dev, (N, M), "bf16")
    kernels.gelu_bwd(q, pre, pre, ref, ref_t)  # the product times GELU'(pre), pre being the product
    kernels.gemm_bf16_gelu_bwd(q, ta, tb, pre, da, da_t)
    assert np.array_equal(da.numpy(q), ref.numpy(q)) and np.array_equal(da_t.numpy(q), ref_t.numpy(q))
    for t in (ta, tb, pre, da, da_t, ref, ref_t):
        t.free()

"""Products with a side below 128 (gemm_skinny.h): every tile count of the short side and both of the
long one, one and several K steps per wave, K that ends inside a step or inside a 16-byte load, the
short side first and second, row-major and packed weights, every epilogue.

f32 results against f64: K products of bf16 values added in f32 in some order, so within
K 2^-24 sum|a||b| (the any-order bound); int8 results bit for bit."""
import numpy as np
import pytest

from oracle import oracle
from vernondsl_amd import _lib, kernels, rng
from vernondsl_amd._lib import call
from vernondsl_amd.rhi import Tensor

pytestmark = pytest.mark.gpu
F32, BF16 = 0, 1

# (M, N, K): 16, 32, 64 and 128 rows in one block and one more row than a tile; wide and narrow long
# sides; 8 and 16 waves; K below one step, of one step, ragged in the step, in the load (odd)
NT = [(1, 1, 8), (1, 5, 16), (8, 96, 256), (16, 33, 32), (17, 64, 2048), (31, 100, 2056), (33, 200, 72), (64, 130, 13),
      (65, 129, 300), (127, 127, 257), (127, 8192, 40), (3, 8200, 2080), (300, 10, 1000), (129, 1, 784), (2000, 64, 2049),
      (1000, 100, 4096), (10, 1000, 300), (24, 9000, 96)]


def operands(M, N, K, seed):
    a = rng.f32_to_bf16(rng.uniform(seed, M * K, -1, 1)).reshape(M, K)
    b = rng.f32_to_bf16(rng.uniform(seed + 1, N * K, -1, 1)).reshape(N, K)
    return a, b


@pytest.mark.parametrize("M,N,K", NT)
def test_row_major(dev, q, M, N, K):
    a, b = operands(M, N, K, M + 3 * N + 7 * K)
    ta, tb = Tensor.from_numpy(dev, q, a, "bf16"), Tensor.from_numpy(dev, q, b, "bf16")
    out, pre, act = Tensor(dev, (M, N), "f32"), Tensor(dev, (M, N), "f32"), Tensor(dev, (M, N), "bf16")
    for t in (out, pre):
        t.buffer.fill_u32(q, 0x7FC00000)
    kernels.gemm_bf16(q, ta, tb, out, False, True)
    kernels.gemm_bf16(q, ta, tb, act, False, True, _lib.EPI_GELU, pre)
    af, bf = rng.bf16_to_f32(a).astype(np.float64), rng.bf16_to_f32(b).astype(np.float64)
    got = out.numpy(q)
    assert np.all(np.abs(got - af @ bf.T) <= K * 2.0 ** -24 * (np.abs(af) @ np.abs(bf).T))
    assert np.array_equal(pre.numpy(q), got)
    g = Tensor(dev, (M, N), "bf16")
    kernels.gelu_fwd(q, out, g)  # GELU of the same f32 values, its own rounding: one bf16 ulp
    x, y = rng.bf16_to_f32(act.numpy(q)), rng.bf16_to_f32(g.numpy(q))
    assert np.all(np.abs(x - y) <= 2.0 ** -7 * np.abs(y) + 1e-30)
    for t in (ta, tb, out, pre, act, g):
        t.free()


@pytest.mark.parametrize("M,N,K", [(1, 32, 256), (8, 96, 4096), (20, 8192, 256), (32, 544, 512), (31, 96, 512), (127, 32, 2304), (16, 16384, 512), (17, 16416, 512), (24, 65536, 256), (9, 65536, 256),
                                   (300, 32, 2048), (2000, 32, 256)])
def test_packed_equals_row_major(dev, q, M, N, K):
    """Packed weights, with every epilogue, against the row-major form and the separate ops, bit for
    bit (every output is one chain of MFMAs over K in all of them)."""
    a, b = operands(M, N, K, M + N + K)
    ta, tb, tbp = Tensor.from_numpy(dev, q, a, "bf16"), Tensor.from_numpy(dev, q, b, "bf16"), Tensor(dev, (N, K), "bf16")
    kernels.pack_bf16_weights(q, tb, tbp)
    f = [Tensor(dev, (M, N), "f32") for _ in range(5)]
    h = [Tensor(dev, (M, N), "bf16") for _ in range(6)]
    ht = [Tensor(dev, (N, M), "bf16") for _ in range(3)]
    kernels.gemm_bf16(q, ta, tb, f[0], False, True)
    kernels.gemm_bf16_packed(q, ta, tbp, f[1])
    assert np.array_equal(f[0].numpy(q), f[1].numpy(q))
    for epi in (_lib.EPI_GELU, _lib.EPI_RELU):
        kernels.gemm_bf16(q, ta, tb, h[0], False, True, epi, f[2])
        kernels.gemm_bf16_packed(q, ta, tbp, h[1], epi, f[3])
        assert np.array_equal(h[0].numpy(q), h[1].numpy(q)) and np.array_equal(f[2].numpy(q), f[3].numpy(q))
    kernels.gemm_bf16_packed(q, ta, tbp, h[1], _lib.EPI_GELU_DERIV, f[4])  # GELU'(pre) in f[4]
    kernels.gemm_bf16_packed(q, ta, tbp, h[0], _lib.EPI_GELU, f[2])
    assert np.array_equal(h[0].numpy(q), h[1].numpy(q))
    kernels.gelu_bwd(q, f[0], f[0], h[2], ht[0])  # dL/dy * GELU'(pre) with dL/dy = pre = the product
    kernels.gemm_bf16_gelu_bwd(q, ta, tb, f[0], h[3], ht[1])
    kernels.gemm_bf16_gelu_bwd(q, ta, tbp, f[0], h[4], ht[2], packed=True)
    kernels.gemm_bf16_mul_packed(q, ta, tbp, f[4], h[5])
    ref, ref_t = h[2].numpy(q), ht[0].numpy(q)
    for t in h[3:]:
        assert np.array_equal(t.numpy(q), ref)
    for t in ht[1:]:
        assert np.array_equal(t.numpy(q), ref_t)
    for t in [ta, tb, tbp] + f + h + ht:
        t.free()


# every configuration of the chain (1, 2 and 4 row tiles, 1 and 2 column tiles; one stage, several and a
# part; K that ends inside a step), waves that load for themselves (K up to 128, 256 on a long side; one
# and two row tiles; a ragged last block), both orders of the short side, and the limits of the rules:
# 16 / 17, 32 / 33 and 127 rows, 8192 and 16384 columns
SAME = [(1, 40, 8), (16, 512, 300), (5, 1000, 520), (17, 96, 1024), (32, 257, 2048), (16, 8200, 160), (32, 8192, 128), (17, 8193, 136),
        (9, 65537, 256), (31, 65536, 72), (33, 96, 1040), (127, 500, 304), (64, 8192, 136), (40, 4200, 264), (300, 10, 1000),
        (9000, 20, 64), (5000, 7, 40), (2000, 100, 712), (1, 1, 4096)]


@pytest.mark.parametrize("M,N,K", SAME)
def test_same_bits_on_every_path(dev, q, M, N, K):
    """A short-side product equals the tile kernels' bit for bit, in all four layouts; so does each row on
    its own (one row's result does not depend on the batch)."""
    a, b = operands(M, N, K, M + 5 * N + K)

    def product(x, y, ta, tb, config=-1):
        m, n = len(x), len(y)
        call("vdsl_debug_gemm_config", config)
        try:
            t = [Tensor.from_numpy(dev, q, np.ascontiguousarray(x.T) if ta else x, "bf16"),
                 Tensor.from_numpy(dev, q, y if tb else np.ascontiguousarray(y.T), "bf16"), Tensor(dev, (m, n), "f32"),
                 Tensor(dev, (max(1, kernels.gemm_bf16_workspace_bytes(ta, tb, m, n, K)),), "i8")]
            t[2].buffer.fill_u32(q, 0x7FC00000)
            kernels.gemm_bf16(q, t[0], t[1], t[2], ta, tb, _lib.EPI_NONE, None, t[3])
            out = t[2].numpy(q)
        finally:
            call("vdsl_debug_gemm_config", -1)
        for v in t:
            v.free()
        return out

    got = product(a, b, False, True)
    if K % 8 == 0:
        assert np.array_equal(got, product(a, b, False, True, config=0))
    for ta, tb in ((False, False), (True, False), (True, True)):
        assert np.array_equal(got, product(a, b, ta, tb)), (ta, tb)
    big = np.concatenate([a] * (200 // M + 1)) if M < 200 else a  # the same rows in a batch past the limit
    assert np.array_equal(got, product(big, b, False, True)[:M])
    assert np.array_equal(got[M // 2:M // 2 + 1], product(a[M // 2:M // 2 + 1], b, False, True))


@pytest.mark.parametrize("M,N,K,packed", [(1, 32, 512, True), (8, 8192, 512, True), (33, 96, 4608, True), (100, 1024, 1024, True),
                                          (300, 64, 512, True), (1, 1, 16, False), (5, 37, 80, False), (17, 8200, 272, False),
                                          (127, 130, 4112, False), (500, 3, 64, False), (64, 1000, 4096, False),
                                          # past the rule's long sides: the tiles, and activations long
                                          (8, 16400, 64, False), (17, 8208, 528, False), (16400, 17, 256, False)])
def test_int8(dev, q, M, N, K, packed):
    r = np.random.default_rng(M * 5 + N + K)
    xq = r.integers(-127, 128, (M, K)).astype(np.int8)
    w = r.integers(-127, 128, (N, K)).astype(np.int8)
    xs, ws = r.uniform(0.01, 0.1, M).astype(np.float32), r.uniform(0.005, 0.02, N).astype(np.float32)
    t = [Tensor.from_numpy(dev, q, v) for v in (xq, xs, w, ws)]
    for dt, relu in (("bf16", True), ("f32", False)):
        y, acc = Tensor(dev, (M, N), dt), Tensor(dev, (M, N), "i32")
        if packed:
            wp = Tensor(dev, (N, K), "i8")
            kernels.pack_w8a8_weights(q, t[2], wp)
            need = kernels.gemm_w8a8_packed_workspace_bytes(M, N, K)
            work = Tensor(dev, (max(1, need),), "i8")
            kernels.gemm_w8a8_packed(q, t[0], t[1], wp, t[3], y, relu, acc, work if need else None)
            wp.free()
        else:
            need = kernels.gemm_w8a8_workspace_bytes(M, N, K)
            work = Tensor(dev, (max(1, need),), "i8")
            kernels.gemm_w8a8(q, t[0], t[1], t[2], t[3], y, relu, acc, work if need else None)
        ry, racc = oracle.gemm_w8a8(xq, xs, w, ws, out_dtype=BF16 if dt == "bf16" else F32, relu=relu, want_acc=True)
        assert np.array_equal(acc.numpy(q), racc) and np.array_equal(y.numpy(q), ry)
        for v in (y, acc, work):
            v.free()
    for v in t:
        v.free()


def test_nan_next_to_k_ends(dev, q):
    """A NaN at the start of a row reaches that row only, though the previous row's last K step reads it."""
    M, N, K = 5, 20, 45
    a, b = operands(M, N, K, 77)
    a[3, 0] = 0x7FC0
    b[11, 0] = 0x7FC0
    for x, y in ((a, b), (b, a)):
        tx, ty, out = Tensor.from_numpy(dev, q, x, "bf16"), Tensor.from_numpy(dev, q, y, "bf16"), Tensor(dev, (len(x), len(y)), "f32")
        kernels.gemm_bf16(q, tx, ty, out, False, True)
        nan = np.isnan(out.numpy(q))
        want = np.zeros_like(nan)
        want[3 if x is a else 11, :] = True
        want[:, 11 if x is a else 3] = True
        assert np.array_equal(nan, want)
        for t in (tx, ty, out):
            t.free()


@pytest.mark.parametrize("M,N,K", [(33, 64, 256), (64, 1024, 512), (100, 96, 512), (130, 4096, 256), (300, 2080, 256), (500, 4096, 512),
                                   (1000, 2048, 256), (2000, 64, 256)])
def test_packed_tiles(dev, q, M, N, K):
    """Every tile size of the packed product (32 x 64 to 128 x 256, whole and ragged) with every epilogue,
    bit for bit against the row-major tiles and the separate ops."""
    a, b = operands(M, N, K, M * 3 + N + K)
    ta, tb, tbp = Tensor.from_numpy(dev, q, a, "bf16"), Tensor.from_numpy(dev, q, b, "bf16"), Tensor(dev, (N, K), "bf16")
    kernels.pack_bf16_weights(q, tb, tbp)
    f = [Tensor(dev, (M, N), "f32") for _ in range(4)]
    h = [Tensor(dev, (M, N), "bf16") for _ in range(6)]
    ht = [Tensor(dev, (N, M), "bf16") for _ in range(3)]
    kernels.gemm_bf16(q, ta, tb, f[0], False, True)
    kernels.gemm_bf16_packed(q, ta, tbp, f[1])
    got = f[0].numpy(q)
    af, bf = rng.bf16_to_f32(a).astype(np.float64), rng.bf16_to_f32(b).astype(np.float64)
    assert np.all(np.abs(got - af @ bf.T) <= K * 2.0 ** -24 * (np.abs(af) @ np.abs(bf).T))
    assert np.array_equal(got, f[1].numpy(q))
    kernels.gemm_bf16(q, ta, tb, h[0], False, True, _lib.EPI_GELU, f[1])
    kernels.gemm_bf16_packed(q, ta, tbp, h[1], _lib.EPI_GELU, f[2])
    kernels.gemm_bf16_packed(q, ta, tbp, h[2], _lib.EPI_GELU_DERIV, f[3])
    ref = h[0].numpy(q)
    assert np.array_equal(f[2].numpy(q), got) and np.array_equal(h[1].numpy(q), ref) and np.array_equal(h[2].numpy(q), ref)
    kernels.gelu_bwd(q, f[0], f[0], h[3], ht[0])
    kernels.gemm_bf16_gelu_bwd(q, ta, tbp, f[0], h[4], ht[1], packed=True)
    kernels.gemm_bf16_mul_packed(q, ta, tbp, f[3], h[5], ht[2])
    for x, y in ((h[4], h[3]), (h[5], h[3]), (ht[1], ht[0]), (ht[2], ht[0])):
        assert np.array_equal(x.numpy(q), y.numpy(q))
    for t in [ta, tb, tbp] + f + h + ht:
        t.free()

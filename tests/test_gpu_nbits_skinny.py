"""The few-row MatMulNBits kernel where it can go wrong: every row layout at its
edges (one, two and three split terms, several row groups), ragged K (a chunk
cut short, an odd K, a block longer than K) and N, every block size class, K
slices, and activations that are not 16-byte aligned.

Bar as in test_gpu_mmnb.py: normwise 1e-5 against the oracle and
gamma_{K+2} sum|a||W| against the 64-bit product; reruns give the same bits.
"""
import ctypes
import os

import numpy as np
import pytest

from oracle import nbits_ex as X
from oracle import refcpu
from onnx_runtime_dart_amd import _lib, ops, synth
from onnx_runtime_dart_amd._lib import check
from tests.helpers import kernels_of, normwise_rel_err

pytestmark = pytest.mark.gpu

U = 2.0 ** -24

CASES = [
    # m, k, n, block, zp
    (2, 512, 33, 16, True),        # one chunk, one segment per k wave
    (5, 1001, 70, 32, True),       # odd K
    (8, 96, 1, 64, False),         # last row of the three-term layout, one column
    (9, 1000, 3001, 32, True),     # first row of the two-term layout, K % 8 == 0
    (16, 2048, 130, 128, True),    # four chunks
    (17, 520, 64, 16, True),       # first row of the two-pass layout, 8 k in chunk 2
    (32, 4096, 100, 32, True),     # K slices
    (6, 5120, 65, 256, False),     # K slices of uneven length
    (33, 1024, 65, 32, True),      # two row groups
    (200, 640, 96, 64, True),      # seven row groups
    (70, 4096, 64, 128, False),    # row groups with K slices
    (4, 300, 40, 1024, True),      # a block longer than K
    (3, 2500, 31, 16, False),
    (3, 859, 33, 128, False),      # rows of no alignment: K % 4 = 3, 2, 1
    (20, 1514, 65, 32, True),
    (54, 2001, 64, 128, False),
    (40, 2000, 2100, 16, True),    # two row groups, four chunks in 32-column workgroups
    (2, 5, 7, 16, True),
    (4, 3, 5, 16, False),          # fewer than four values
    (5, 2000, 130, 32, True),
    (4, 2000, 130, 32, True),      # the multi-row GEMV: four rows, and its longest rows
    (2, 16384, 65, 64, False),
    (18, 8192, 4100, 64, True),    # six chunks a slice
    (18, 4700, 8260, 64, True),    # beyond a workgroup's chunks: the GEMM
    (300, 256, 1030, 32, False),
]


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("m,k,n,block,zp", CASES)
def test_few_rows(m, k, n, block, zp, offset):
    ctx = _lib.default_context()
    p = synth.mmnb_problem(m, k, n, block, zp, seed=m + k + n, outlier_frac=0.01)
    pack = ops.pack_nbits(p.b_q, p.scales, p.zero_points, k=k, n=n, bits=4, block_size=block,
                          ctx=ctx)
    # offset 1: rows that start 4 bytes past a 16-byte boundary
    host = np.zeros(m * k + offset, np.float32)
    host[offset:] = p.a.ravel()
    da, dy = ctx.to_device(host), ctx.alloc(m * n * 4)
    try:
        def run():
            dy.upload(np.full(m * n, np.nan, np.float32))
            check(ctx.lib.mmnb_matmul_nbits_dev(
                ctx.handle, pack.handle, ctypes.c_void_p(da.ptr.value + 4 * offset), m, dy.ptr))
            ctx.synchronize()
            return dy.numpy(np.float32, (m, n))
        y = run()
        ref = refcpu.matmul_nbits(p.a, p.b_q, p.scales, p.zero_points, k, n, 4, block, threads=8)
        assert normwise_rel_err(y, ref) <= 1e-5
        y64, absdot = refcpu.matmul_nbits_f64(p.a, p.b_q, p.scales, p.zero_points, k, n, block)
        gam = (k + 2) * U / (1 - (k + 2) * U)
        assert np.all(np.abs(y - y64) <= gam * absdot + 1e-30)
        np.testing.assert_array_equal(run(), y)
    finally:
        da.free()
        dy.free()
        pack.free()


def _spread(p, rng, ratios):
    """Rows whose magnitudes differ by powers of `ratios` inside 512 k, the large ones over
    weights that equal their zero point, so that no large product hides a lost small one."""
    n, nb, half = p.b_q.shape
    zi = np.arange(n * nb)
    z = np.full(n * nb, 8, np.uint8) if p.zero_points is None else \
        (p.zero_points[zi >> 1] >> (4 * (zi & 1))) & 15
    z = z.astype(np.uint8).reshape(n, nb)
    for r, ratio in enumerate(ratios):
        for k in rng.choice(p.k, max(1, p.k // 300), replace=False):
            p.a[:, k] = 0.0
            p.a[r, k] = ratio
            b, i, sh = k // p.block, k % p.block // 2, 4 * (k & 1)
            p.b_q[:, b, i] = (p.b_q[:, b, i] & (0xF0 >> sh)) | (z[:, b] << sh)


@pytest.mark.parametrize("m,k,n,block,zp,ratios", [
    (5, 512, 40, 32, True, (1e6, 1e8, 1e12, 1e20, 1e38)),     # one piece, every row another
    (8, 4096, 70, 128, False, (1e9, 1.0, 1e38)),              # K slices; rows without
    (2, 1999, 33, 64, True, (1e15,)),                         # a cut chunk, K % 4 = 3
    (6, 1000, 3001, 32, False, (1e11, 1e13, 1e10)),           # 32-column workgroups
    (3, 20, 9, 16, True, (1e12, 1e30)),
    (8, 6000, 9000, 16, False, (1e13, 1e25)),                 # several chunks without slices
])
def test_magnitudes_of_any_range_in_a_row(m, k, n, block, zp, ratios):
    ctx = _lib.default_context()
    p = synth.mmnb_problem(m, k, n, block, zp, seed=5 * m + k)
    rng = np.random.default_rng(k)
    p.a[m - 1, 1::2] *= np.float32(2.0) ** rng.integers(-140, 30, p.a[m - 1, 1::2].shape)
    _spread(p, rng, ratios)
    y = ops.op_matmul_nbits(p.a, p.b_q, p.scales, p.zero_points, k=k, n=n, bits=4,
                            block_size=block, ctx=ctx)
    y64, absdot = refcpu.matmul_nbits_f64(p.a, p.b_q, p.scales, p.zero_points, k, n, block)
    gam = (k + 2) * U / (1 - (k + 2) * U)
    assert np.all(np.abs(y - y64) <= gam * absdot + 1e-30)


@pytest.fixture(scope="module")
def lean_ctx():
    # packs without the few-row kernel's copy of the weights
    saved = os.environ.get("MMNB_FEW_ROW_COPY")
    os.environ["MMNB_FEW_ROW_COPY"] = "0"
    try:
        c = _lib.Context(0)
    finally:
        if saved is None:
            os.environ.pop("MMNB_FEW_ROW_COPY", None)
        else:
            os.environ["MMNB_FEW_ROW_COPY"] = saved
    yield c
    c.close()


@pytest.mark.parametrize("m,k,n,bits,block,zp,bias", [
    (2, 1000, 65, 4, 32, True, False),
    (5, 9000, 40, 4, 64, False, False),    # five rows do not fit LDS
    (8, 4096, 130, 4, 128, True, True),
    (7, 512, 33, 4, 16, False, True),      # 4 + 3
    (9, 2048, 70, 4, 32, True, False),     # the GEMM
    (6, 1000, 50, 8, 32, False, True),
    (3, 700, 41, 8, 64, True, True),
    (20, 640, 64, 8, 32, False, False),
])
def test_packs_without_the_copy(lean_ctx, m, k, n, bits, block, zp, bias):
    rng = np.random.default_rng(m + k)
    nb = -(-k // block)
    b = rng.integers(0, 256, (n, nb, block * bits // 8)).astype(np.uint8)
    s = rng.uniform(0.002, 0.02, n * nb).astype(np.float32)
    z = rng.integers(0, 256, n * nb if bits == 8 else (n * nb + 1) // 2).astype(np.uint8)
    z = z if zp else None
    bv = rng.standard_normal(n).astype(np.float32) if bias else None
    a = rng.standard_normal((m, k)).astype(np.float32)
    y, size = [], []
    for ctx in (lean_ctx, _lib.default_context()):
        pack = ops.pack_nbits_ex(b, s, z, None, bv, k=k, n=n, bits=bits, block_size=block, ctx=ctx)
        try:
            y.append(np.empty((m, n), np.float32))
            check(ctx.lib.mmnb_matmul_nbits(ctx.handle, pack.handle, _lib.ptr(a), m,
                                            _lib.ptr(y[-1])))
            size.append(pack.device_bytes)
        finally:
            pack.free()
    assert size[1] - size[0] >= n * nb * block * bits // 8
    y64, _ = X.matmul_nbits_ex_f64(a, b, s, z, None, bv, k, n, bits, block)
    q = X.unpack_q(b, k, n, bits, block).astype(np.float64)
    gi = np.arange(k) // block
    # the bound of tests/test_gpu_nbits_ex.py (8 bits: planes of 16 hi and lo)
    part = np.abs(q) + np.abs(X.zero_points_per_block(z, n, nb, bits)[:, gi])
    part = (part + (272.0 if bits == 8 else 0.0)) * s.astype(np.float64).reshape(n, nb)[:, gi]
    kk = (2 if bits == 8 else 1) * k + nb + 4
    scale = np.abs(a.astype(np.float64)) @ part.T + (0 if bv is None else np.abs(bv.astype(float)))
    for v in y:
        assert np.all(np.abs(v - y64) <= kk * U / (1 - kk * U) * scale + 1e-30)


@pytest.mark.parametrize("m,k,n,bits,block,kernel", [
    (1, 512, 64, 4, 32, "k_gemv_valu"), (1, 512, 64, 8, 32, "k_gemv8"),
    (2, 2048, 256, 4, 32, "k_gemv_lds"), (4, 2048, 256, 4, 32, "k_gemv_lds"),
    (2, 8192, 4096, 4, 128, "k_gemv_lds"), (5, 2048, 256, 4, 32, "k_nbits_skinny"),
    (3, 4096, 8192, 4, 16, "k_nbits_skinny"), (2, 4096, 14336, 4, 32, "k_nbits_skinny"),
    (16, 4096, 4096, 4, 32, "k_nbits_skinny"), (32, 4096, 256, 4, 32, "k_nbits_skinny"),
    (20, 4096, 256, 4, 16, "k_nbits_skinny"), (20, 8192, 4096, 4, 16, "k_nbits_skinny"),
    (20, 8192, 8320, 4, 16, "k_gemm_mfma"),
    (64, 2048, 4096, 4, 16, "k_nbits_skinny"), (64, 4096, 4096, 4, 16, "k_gemm_mfma"),
    (17, 8192, 16384, 4, 128, "k_gemm_mfma"), (64, 2048, 2048, 4, 32, "k_nbits_skinny"),
    (256, 64, 4096, 4, 32, "k_gemm_mfma"), (256, 256, 4096, 4, 32, "k_nbits_skinny"),
    (100, 4096, 4096, 4, 32, "k_gemm_mfma"),
])
def test_kernel_of_a_call(m, k, n, bits, block, kernel):
    ctx = _lib.default_context()
    nb = -(-k // block)
    pack = ops.pack_nbits_ex(np.full((n, nb, block * bits // 8), 0x77, np.uint8),
                             np.ones(n * nb, np.float32), k=k, n=n, bits=bits, block_size=block,
                             ctx=ctx)
    da, dy = ctx.to_device(np.zeros((m, k), np.float32)), ctx.alloc(m * n * 4)
    try:
        assert kernel in kernels_of(ctx, lambda: check(ctx.lib.mmnb_matmul_nbits_dev(
            ctx.handle, pack.handle, da.ptr, m, dy.ptr)))
    finally:
        da.free()
        dy.free()
        pack.free()

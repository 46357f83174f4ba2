"""GPU parity of extended packs that need no correction pass: 8-bit weights with integer
zero points (k_gemv8 for one row, else the planes through the few-row kernel and the
GEMM) and 4-bit weights with a bias, at the edges of chunks, planes and column groups.

Bar: |y - y64| <= gamma_{K + n_blocks + 4} * sum|a| |q - zp| scale (+ |bias|) for one
row, whose kernels form q - zp exactly (no hi/lo split and no correction); the bound of
tests/test_gpu_nbits_ex.py for more rows.
"""
import numpy as np
import pytest

from oracle import nbits_ex as X
from onnx_runtime_dart_amd import _lib, ops

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def _problem(m, k, n, bits, bs, zp, bias, seed):
    rng = np.random.default_rng(seed)
    nb = (k + bs - 1) // bs
    b = rng.integers(0, 256, (n, nb, bs * bits // 8)).astype(np.uint8)
    s = rng.uniform(0.002, 0.02, n * nb).astype(np.float32)
    z = None
    if zp:
        z = rng.integers(0, 256, n * nb if bits == 8 else (n * nb + 1) // 2).astype(np.uint8)
    bv = rng.standard_normal(n).astype(np.float32) if bias else None
    a = rng.standard_normal((m, k)).astype(np.float32)
    return a, b, s, z, bv, nb


@pytest.mark.parametrize("m,k,n,bits,bs,zp,bias", [
    (1, 16, 1, 8, 16, True, False),        # one block, one column
    (1, 3, 5, 8, 16, True, True),          # fewer than four values
    (1, 2907, 130, 8, 64, False, True),    # K % 4 = 3, 2, 1
    (1, 1014, 66, 8, 32, True, False),
    (1, 4165, 9, 8, 128, True, True),
    (1, 100, 5, 8, 16, False, True),       # ragged K, blocks of 16 (padded planes)
    (1, 96, 130, 8, 32, True, True),       # an odd number of blocks
    (1, 2048, 67, 8, 32, False, False),
    (1, 4096, 64, 8, 128, False, True),    # one chunk per lane in every wave
    (1, 4160, 9, 8, 64, True, False),      # a second pass over K
    (1, 1000, 4096, 8, 128, True, True),   # a partial block
    (3, 96, 70, 8, 32, True, True),        # padded planes through the few-row kernel
    (100, 96, 70, 8, 32, True, False),     # ... and through the GEMM
    (2, 36, 33, 8, 16, True, True),        # rows that are not whole 8-k runs
    (8, 1000, 130, 8, 128, True, True),    # the second plane inside a 512-k piece
    (16, 4096, 96, 8, 32, False, True),    # K slices
    (20, 700, 65, 8, 64, True, False),
    (600, 1000, 520, 8, 128, True, True),  # the GEMM, tiles with and without K groups
    (70, 4160, 300, 8, 64, False, True),   # ... its K slices
    (5, 1000, 301, 4, 32, True, True),     # 4-bit weights with a bias, several rows
    (24, 4096, 100, 4, 128, False, True),
    (2, 1024, 70, 4, 16, True, True),      # ... through the multi-row GEMV
    (4, 2048, 77, 4, 32, True, True),
    (5, 2000, 300, 4, 128, False, True),   # five rows: the few-row kernel
    (2, 1000, 90, 8, 32, True, True),      # 8-bit planes, gathered for it
    (4, 3, 9, 8, 16, False, True),         # fewer than four values: row by row, the GEMM
    (11, 2, 9, 8, 16, True, False),
    (9, 3, 9, 4, 16, True, True),
    (130, 2048, 300, 4, 64, True, True),
    (1, 1000, 301, 4, 32, True, True),     # ... and one
    (1, 4160, 3, 4, 128, False, True),
])
def test_packs_without_a_correction(m, k, n, bits, bs, zp, bias):
    a, b, s, z, bv, nb = _problem(m, k, n, bits, bs, zp, bias, m + k + n)
    y = ops.op_matmul_nbits_ex(a, b, s, z, None, bv, k=k, n=n, bits=bits, block_size=bs,
                               ctx=_lib.default_context())
    y64, _ = X.matmul_nbits_ex_f64(a, b, s, z, None, bv, k, n, bits, bs)
    q = X.unpack_q(b, k, n, bits, bs).astype(np.float64)
    zz = X.zero_points_per_block(z, n, nb, bits)
    gi = np.arange(k) // bs
    sc = s.astype(np.float64).reshape(n, nb)[:, gi]
    if m == 1:
        part, kk = np.abs(q - zz[:, gi]) * sc, k + nb + 4
    else:
        part, kk = (np.abs(q) + np.abs(zz[:, gi]) + 272.0) * sc, 2 * k + nb + 4
    scale = np.abs(a.astype(np.float64)) @ part.T
    if bias:
        scale = scale + np.abs(bv.astype(np.float64))
    assert np.all(np.abs(y - y64) <= kk * U / (1 - kk * U) * scale + 1e-30)


def test_non_finite_activations_follow_the_reference():
    a, b, s, z, _, _ = _problem(1, 256, 40, 8, 32, True, False, 3)
    b[:, 0, 7] = z.reshape(40, 8)[:, 0]    # weight 0 under a[7]
    b[20:, 0, 7] ^= 0x55                   # ... and not 0 from column 20 on
    a[0, 7] = np.inf
    y = ops.op_matmul_nbits_ex(a, b, s, z, k=256, n=40, bits=8, block_size=32,
                               ctx=_lib.default_context())
    ref = X.matmul_nbits_ex(a, b, s, z, None, None, 256, 40, 8, 32)
    assert np.isnan(ref[0, :20]).all() and np.isinf(ref[0, 20:]).all()
    np.testing.assert_array_equal(np.isnan(y), np.isnan(ref))
    np.testing.assert_array_equal(y[0, 20:], ref[0, 20:])

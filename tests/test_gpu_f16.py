"""Products of more than 16 tokens by F16 weights on the f16 matrix instruction, the activations in three f16 parts under a
factor per 256 columns (csrc/plain_gemm.inc), against float64.

Tolerances as in test_gpu_parity.py: the proven bound of any f32 summation order and the reference's observed envelope,
both relative to sum |w x| (langtax/src/simd/tests.rs:18-91)."""
import numpy as np
import pytest

import cases as K

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu(pkg):
    g = pkg.HipGemv(0)
    yield g
    g.close()


def _check(gpu, w, x):
    rows, cols = w.shape
    tokens = x.shape[0]
    m = gpu.upload_packed(K.F16, rows, cols, np.ascontiguousarray(w).view(np.uint8).reshape(-1))
    y = np.full(tokens * rows, np.nan, np.float32)
    gpu.gemm_resident(m, tokens, x.reshape(-1), y)
    m.close()
    w64, x64 = w.astype(np.float64), x.astype(np.float64)
    err, mag = np.abs(y.reshape(tokens, rows) - x64 @ w64.T), np.abs(x64) @ np.abs(w64).T
    assert np.all(np.isfinite(y))
    assert np.all(err <= K.single_kernel_bound(cols, mag))
    assert np.all(err <= K.observed_envelope_u(cols) * K.U * mag)


# tiles of 32, 64 and 128 tokens (256 rows), their edges, ragged columns, one step and shares of a step or two, blocks of 256 columns
@pytest.mark.parametrize("rows,cols,tokens", [(20, 31, 33), (127, 33, 40), (257, 288, 65), (129, 1000, 64), (300, 2056, 100), (1030, 8200, 130),
                                              (4096, 2048, 257), (2048, 4096, 24), (16, 9000, 40)])
def test_tile_edges(gpu, rows, cols, tokens):
    rng = np.random.default_rng(rows + cols + tokens)
    _check(gpu, rng.normal(0, 0.02, (rows, cols)).astype(np.float16), rng.normal(0, 1, (tokens, cols)).astype(np.float32))


@pytest.mark.parametrize("cols", [700, 2048])
def test_numbers_of_every_magnitude(gpu, cols):
    """Subnormal and largest weights; activations that three f16 parts hold, and rows that are taken again in f32."""
    rng = np.random.default_rng(cols)
    rows, tokens = 200, 70
    bits = rng.integers(0, 1 << 16, (rows, cols)).astype(np.uint16)
    bits[(bits & 0x7c00) == 0x7c00] ^= 0x4000  # no infinities or NaN
    bits[:20] &= 0x83ff                        # subnormal rows
    w = bits.view(np.float16)
    x = rng.normal(0, 1, (tokens, cols)).astype(np.float32)
    mant = rng.integers(0, 1 << 23, size=(8, cols)).astype(np.uint32)
    sign = rng.integers(0, 2, size=(8, cols)).astype(np.uint32) << 31
    x[0] = (np.uint32(0x3FFFFFFF) | sign[0]).view(np.float32)
    x[1] = (rng.integers(127 - 60, 127 + 61, size=cols).astype(np.uint32) << 23 | mant[1] | sign[1]).view(np.float32)
    x[2] = ((np.uint32(27) << 23) | mant[2] | sign[2]).view(np.float32)  # 2^-100
    x[3] = ((np.uint32(220) << 23) | mant[3] | sign[3]).view(np.float32)  # 2^93
    x[4, ::3], x[4, 1::3] = 0.0, -0.0
    x[5] = rng.normal(0, 1e-3, cols)
    x[5, 77] = 3.0e4
    x[6] = 0.0
    x[7] = rng.normal(0, 1e-9, cols)
    x[7, cols - 1] = 1.0e4                     # its column's weight may be anything: the others must not be lost beside it
    x[69] = x[1][::-1]
    w[:, cols - 1] = np.where(np.arange(rows) % 2, w[:, cols - 1], np.float16(0.0))
    _check(gpu, w, x)


def test_small_activations_beside_a_few_large_ones_of_zero_weights(gpu):
    """The sum is the small ones' alone: they must not be held to what the large ones allow."""
    rng = np.random.default_rng(3)
    rows, cols, tokens = 140, 1024, 70
    w = rng.normal(0, 0.02, (rows, cols)).astype(np.float16)
    x = np.zeros((tokens, cols), np.float32)
    for g in range(cols // 256):
        at = 256 * g + rng.permutation(256)[:10]
        w[:, at[:7]] = 0
        x[:, at[:7]] = rng.uniform(0.5, 1, (tokens, 7))
        x[:, at[7:]] = rng.normal(0, 2.0 ** -32, (tokens, 3))
    _check(gpu, w, x)

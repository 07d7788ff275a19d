"""Products of more than 16 tokens by F16 weights on the f16 matrix instruction, the activations in three f16 parts under a
factor per 256 columns, and on the f32 instruction where parts or weights do not fit it (csrc/plain_gemm.inc), against float64.

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


# ------------------------------------------------------------------ every activation in all its bits, whatever stands beside it
def _product(gpu, w, x):
    rows, cols = w.shape
    m = gpu.upload_packed(K.F16, rows, cols, np.ascontiguousarray(w).view(np.uint8).reshape(-1))
    y = np.full(x.shape[0] * rows, np.nan, np.float32)
    gpu.gemm_resident(m, x.shape[0], np.ascontiguousarray(x).reshape(-1), y)
    m.close()
    return y.reshape(x.shape[0], rows)


def _spread(kind, rng, shape):
    n = rng.normal(0, 1, shape)
    if kind == "swiglu":
        n = 3 * n / (1 + np.exp(-3 * n)) * 3 * rng.normal(0, 1, shape)
    elif kind == "lognormal":
        n = n * np.exp(2 * rng.normal(0, 1, shape))
    elif kind == "outliers":
        n[:, 5::97] *= 1e5
    elif kind == "decades":  # some in every block of 256 columns lie below what its three parts reach
        n = n * 10.0 ** rng.uniform(-16, 16, shape)
    return n.astype(np.float32)


@pytest.mark.parametrize("large", [1, 7, 8, 20])
@pytest.mark.parametrize("cols,top", [(256, 0), (2100, 0), (2100, 60), (2100, -60), (2100, 126), (17000, 0)])
def test_small_activations_alone_make_the_sum(gpu, large, cols, top):
    """One to five of 256 activations, 2^-13 to 2^-44 below `large` ones whose weights are zero."""
    rng = np.random.default_rng(large + cols + top)
    rows, tokens = 70, 90
    w = rng.normal(0, 0.02, (rows, cols)).astype(np.float16)
    x = np.zeros((tokens, cols))
    for g in range(cols // 256):
        at = 256 * g + rng.permutation(256)[:large + 5]
        x[:, at[:large]] = rng.uniform(0.5, 1, (tokens, large))
        w[:, at[:large]] = 0
        for t in range(tokens):
            n = 1 + t % 5
            x[t, at[large:large + n]] = rng.choice([-1, 1], n) * rng.uniform(0.5, 1, n) * 2.0 ** (-13 - (t + g) % 32)
    x = (x * 2.0 ** top).astype(np.float32)
    y = _product(gpu, w, x)
    w64, x64 = w.astype(np.float64), x.astype(np.float64)
    mag = np.abs(x64) @ np.abs(w64).T
    assert np.all(np.abs(y - x64 @ w64.T) <= K.single_kernel_bound(5 * (cols // 256), mag))  # that many terms are not zero


@pytest.mark.parametrize("other", [1, 5, 9, 20])
@pytest.mark.parametrize("exponent", [0, -6, -13, -20])
def test_subnormal_weights_beside_others(gpu, other, exponent):
    """Two products a row, of the same magnitude or far apart, one of a subnormal weight: neither is held to a normal number's place."""
    rng = np.random.default_rng(40 + other - exponent)
    rows, cols, tokens = 256, 256, 352
    w = np.zeros((rows, cols), np.float16)
    w[:, 0] = rng.choice([1, 3, 1000], rows) * 2.0 ** -24
    w[:, other] = (rng.uniform(1, 2, rows) * 2.0 ** exponent).astype(np.float16)
    x = np.zeros((tokens, cols), np.float32)
    x[:, 0] = 0.75
    x[:, other] = rng.uniform(0.5, 1, tokens) * 2.0 ** -(np.arange(tokens) % 44)
    w64, x64 = w.astype(np.float64), x.astype(np.float64)
    assert np.all(np.abs(_product(gpu, w, x) - x64 @ w64.T) <= K.single_kernel_bound(2, np.abs(x64) @ np.abs(w64).T))


@pytest.mark.parametrize("cols", [700, 2048])
def test_weights_of_every_magnitude(gpu, cols):
    """Every finite f16 number among the weights, few and many of 64 and more (which the scaled weights do not hold)."""
    rng = np.random.default_rng(cols)
    rows, tokens = 300, 70
    w = rng.normal(0, 0.02, (rows, cols)).astype(np.float16)
    bits = rng.integers(0, 0x5400, (200, cols)).astype(np.uint16)  # below 64
    w[:200] = (bits | (rng.integers(0, 2, bits.shape).astype(np.uint16) << 15)).view(np.float16)
    w[::7, 3::11] = rng.uniform(-60000, 60000, w[::7, 3::11].shape)
    w[5, 9], w[40, 0], w[41, cols - 1] = 64, 63.97, -65504
    _check(gpu, w, rng.normal(0, 1, (tokens, cols)).astype(np.float32))


# tiles of 32, 64 and 128 tokens; columns in shares that begin within 256 columns
@pytest.mark.parametrize("kind", ["normal", "swiglu", "lognormal", "outliers", "decades"])
@pytest.mark.parametrize("rows,cols,tokens", [(300, 1000, 40), (512, 512, 100), (2048, 4100, 20), (4096, 2500, 130)])
def test_rows_of_one_weight(gpu, kind, rows, cols, tokens):
    """One product per result: its activation's three exact parts and the sums of shares, a rounding each."""
    rng = np.random.default_rng(rows + cols + tokens)
    x = _spread(kind, rng, (tokens, cols))
    col, weight = rng.integers(0, cols, rows), rng.normal(0, 0.02, rows).astype(np.float16)
    w = np.zeros((rows, cols), np.float16)
    w[np.arange(rows), col] = weight
    exact = x.astype(np.float64)[:, col] * weight.astype(np.float64)
    assert np.all(np.abs(_product(gpu, w, x) - exact) <= 8 * K.U * np.abs(exact))


@pytest.mark.parametrize("kind", ["swiglu", "lognormal", "outliers", "decades"])
# 1003: rows of activations that are aligned to single numbers
@pytest.mark.parametrize("rows,cols,tokens", [(300, 1000, 40), (129, 1003, 33), (1030, 8200, 70), (4096, 2500, 130)])
def test_dense_rows_by_activations_of_wide_range(gpu, kind, rows, cols, tokens):
    rng = np.random.default_rng(rows + cols + tokens)
    _check(gpu, rng.normal(0, 0.02, (rows, cols)).astype(np.float16), _spread(kind, rng, (tokens, cols)))


def test_infinities_and_wide_blocks_stay_in_their_token(gpu):
    rng = np.random.default_rng(8)
    w, x = rng.normal(0, 0.02, (200, 1000)).astype(np.float16), rng.normal(0, 1, (100, 1000)).astype(np.float32)
    clean = _product(gpu, w, x)
    x[3, 100], x[17, 5], x[99, 999] = np.inf, np.nan, -np.inf
    x[40, 300], x[50, :] = 1e-20, x[50, :] * _spread("decades", rng, 1000)
    y = _product(gpu, w, x)
    assert not np.isfinite(y[[3, 17, 99]]).any() and np.isfinite(y[[40, 50]]).all()
    rest = [t for t in range(100) if t not in (3, 17, 99, 40, 50)]
    assert np.array_equal(y[rest], clean[rest])
    w[7, 500] = np.inf  # an infinite weight: its row alone
    y2 = _product(gpu, w, x)
    assert not np.isfinite(y2[:, 7]).any()
    assert np.array_equal(np.delete(y2, 7, 1), np.delete(y, 7, 1), equal_nan=True)

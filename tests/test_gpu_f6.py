"""Products of more than 32 tokens by Q4_0, Q5_0 and Q4_K: both operands as 6-bit floats with block scales
(csrc/f6_gemm.inc), against the oracle's float64 product.

Tolerances as in test_gpu_parity.py: the proven bound of any f32 summation order and the reference's observed envelope,
both relative to sum |w x| (langtax/src/simd/tests.rs:18-91)."""
import numpy as np
import pytest

import cases as K
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu(pkg):
    g = pkg.HipGemv(0)
    yield g
    g.close()


def _product(gpu, ty, rows, cols, x, w):
    m = gpu.upload_packed(ty, rows, cols, w)
    y = np.full(x.shape[0] * rows, np.nan, np.float32)
    gpu.gemm_resident(m, x.shape[0], x.reshape(-1), y)
    m.close()
    return y.reshape(x.shape[0], rows)


def _check(ty, rows, cols, x, w, y):
    exact, mag = O.gemm_f64_mag(ty, cols, x.shape[0], w, x.reshape(-1), rows)
    err = np.abs(y.astype(np.float64) - exact)
    assert np.all(np.isfinite(y))
    # 2^-130 per column and unit of weight: what an activation below 2^-99 is held to
    floor = cols * 2.0 ** -130 * 16 * 64
    assert np.all(err <= K.single_kernel_bound(cols, mag) + floor)
    assert np.all(err <= K.observed_envelope_u(cols) * K.U * mag + floor)


# one group and an odd count of groups (32-column dtypes), whole super-blocks, shared columns; edges of row and token tiles
SHAPES = [(1, 32, 33), (257, 96, 64), (256, 64, 65), (300, 2080, 129), (255, 256, 33), (257, 768, 100), (1000, 4096, 70)]


@pytest.mark.parametrize("ty", [K.Q4_0, K.Q5_0, K.Q4_K], ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("rows,cols,tokens", SHAPES)
def test_tile_edges(gpu, ty, rows, cols, tokens):
    if cols % K.QK[ty]:
        cols = (cols // K.QK[ty] + 1) * K.QK[ty]
    rng = np.random.default_rng(7 * rows + cols + tokens + ty)
    w = K.random_packed(ty, rows, cols, rng)
    x = rng.normal(0, 1, (tokens, cols)).astype(np.float32)
    _check(ty, rows, cols, x, w, _product(gpu, ty, rows, cols, x, w))


@pytest.mark.parametrize("ty", [K.Q4_0, K.Q5_0, K.Q4_K], ids=lambda t: O.TYPE_NAMES[t])
def test_activations_of_every_magnitude(gpu, ty):
    """Groups whose activations six digits hold, groups that are kept as f32 numbers, and both in one tile."""
    rng = np.random.default_rng(91 + ty)
    rows, cols, tokens = 96, 2048, 70
    w = K.random_packed(ty, rows, cols, rng)
    x = rng.normal(0, 1, (tokens, cols)).astype(np.float32)
    mant = rng.integers(0, 1 << 23, size=(8, cols)).astype(np.uint32)
    sign = rng.integers(0, 2, size=(8, cols)).astype(np.uint32) << 31
    x[0] = (np.uint32(0x3FFFFFFF) | sign[0]).view(np.float32)  # every significand bit
    e = rng.integers(127 - 60, 127 + 61, size=cols).astype(np.uint32) << 23
    x[1] = (e | mant[1] | sign[1]).view(np.float32)            # 2^-60 .. 2^60 in every group
    x[2] = ((np.uint32(27) << 23) | mant[2] | sign[2]).view(np.float32)  # 2^-100
    x[3] = ((np.uint32(20) << 23) | mant[3] | sign[3]).view(np.float32)  # 2^-107
    x[4, ::3], x[4, 1::3] = 0.0, -0.0
    x[5] = rng.normal(0, 1e-3, cols)
    x[5, 777] = 3.0e4                                          # one large among small ones
    x[6] = 0.0
    x[7] = (x[7] * 2.0 ** 90).astype(np.float32)
    x[40] = x[1][::-1]
    x[69] = x[5][::-1]                                         # the last token of a partial tile
    _check(ty, rows, cols, x, w, _product(gpu, ty, rows, cols, x, w))


@pytest.mark.parametrize("ty", [K.Q4_0, K.Q5_0], ids=lambda t: O.TYPE_NAMES[t])
def test_small_activations_beside_a_few_large_ones_of_zero_weights(gpu, ty):
    """The sum is the small ones' alone: they must not be held to what the large ones allow."""
    rng = np.random.default_rng(23 + ty)
    cols, tokens = 512, 40
    w = K.random_packed(ty, 1, cols, rng)
    w32 = O.dequant(ty, cols, w, 1).reshape(-1, 32)
    x = np.zeros((tokens, cols), np.float32)
    for g in range(cols // 32):
        zero, rest = np.flatnonzero(w32[g] == 0), np.flatnonzero(w32[g] != 0)
        at = rng.permutation(rest)[:3]
        x[:, 32 * g + at] = rng.normal(0, 2.0 ** -22, (tokens, 3))
        x[:, 32 * g + zero[:7]] = rng.uniform(0.5, 1, (tokens, len(zero[:7])))
    _check(ty, 1, cols, x, w, _product(gpu, ty, 1, cols, x, w))


@pytest.mark.parametrize("ty", [K.Q4_0, K.Q4_K], ids=lambda t: O.TYPE_NAMES[t])
def test_infinities_stay_in_their_token(gpu, ty):
    rng = np.random.default_rng(5)
    rows, cols, tokens = 64, 512, 40
    w = K.random_packed(ty, rows, cols, rng)
    x = rng.normal(0, 1, (tokens, cols)).astype(np.float32)
    clean = _product(gpu, ty, rows, cols, x, w)
    x[3, 100], x[17, 5], x[39, 511] = np.inf, np.nan, -np.inf
    y = _product(gpu, ty, rows, cols, x, w)
    hit = [3, 17, 39]
    rest = [t for t in range(tokens) if t not in hit]
    assert not np.isfinite(y[hit]).any()
    assert np.array_equal(y[rest], clean[rest])

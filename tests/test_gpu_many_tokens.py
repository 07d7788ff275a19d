"""Products of more than 32 tokens by block-quantized matrices: every activation is held in all its bits, whatever stands
beside it (csrc/gemm_kernels.inc), against the oracle's float64 product.

Tolerances as in test_gpu_parity.py: the proven bound of any f32 summation order and the reference's observed envelope,
both relative to sum |w x| (langtax/src/simd/tests.rs:18-91)."""
import importlib

import numpy as np
import pytest

import cases as K
import oracle as O

pytestmark = pytest.mark.gpu

QUANTIZED = [K.Q4_0, K.Q5_0, K.Q5_1, K.Q8_0, K.Q4_K, K.Q6_K]


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


@pytest.mark.parametrize("ty", QUANTIZED, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("rows,cols,tokens", SHAPES)
def test_tile_edges(gpu, ty, rows, cols, tokens):
    if cols % K.QK[ty]:
        cols = (cols // K.QK[ty] + 1) * K.QK[ty]
    rng = np.random.default_rng(7 * rows + cols + tokens + ty)
    w = K.random_packed(ty, rows, cols, rng)
    x = rng.normal(0, 1, (tokens, cols)).astype(np.float32)
    _check(ty, rows, cols, x, w, _product(gpu, ty, rows, cols, x, w))


@pytest.mark.parametrize("ty", QUANTIZED, ids=lambda t: O.TYPE_NAMES[t])
def test_activations_of_every_magnitude(gpu, ty):
    """2^-107 to 2^93, every significand bit, one large among small ones, zeros; also in the last token of a partial tile."""
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


def _keep_columns(ty, rows, cols, w, keep):
    """A copy of the packed rows in which the weights of all columns but keep[row] (bool, rows x cols) are zero."""
    b = w.copy().reshape(rows, cols // K.QK[ty], K.BLOCK[ty])
    zero = ~keep.reshape(rows, cols // K.QK[ty], K.QK[ty])

    def nibbles(at, mask, code):
        """Code `code` into the low nibbles of bytes at.. where mask[0], into the high ones where mask[1]."""
        v = b[:, :, at:at + mask[0].shape[-1]]
        v[mask[0]] = v[mask[0]] & 0xF0 | code
        v[mask[1]] = v[mask[1]] & 0x0F | code << 4

    if ty == K.Q8_0:
        b[:, :, 2:][zero] = 0
    elif ty == K.Q4_0:
        nibbles(2, (zero[..., :16], zero[..., 16:]), 8)
    elif ty in (K.Q5_0, K.Q5_1):
        off = 2 if ty == K.Q5_0 else 4
        nibbles(off + 4, (zero[..., :16], zero[..., 16:]), 0)
        bits = np.packbits(zero, axis=-1, bitorder="little")
        if ty == K.Q5_0:
            b[:, :, off:off + 4] |= bits  # code 16
        else:
            b[:, :, off:off + 4] &= ~bits
            b[:, :, 2:4] = 0              # no offset
    elif ty == K.Q4_K:
        b[:, :, 2:4] = 0
        for n in range(4):
            nibbles(16 + 32 * n, (zero[..., 64 * n:64 * n + 32], zero[..., 64 * n + 32:64 * n + 64]), 0)
    else:
        for n in range(2):
            z = zero[..., 128 * n:128 * n + 128].reshape(rows, -1, 4, 32)
            for k in range(2):
                nibbles(64 * n + 32 * k, (z[:, :, k], z[:, :, k + 2]), 0)
            high = b[:, :, 128 + 32 * n:160 + 32 * n]
            for q in range(4):
                high[z[:, :, q]] = high[z[:, :, q]] & ~np.uint8(3 << 2 * q) | np.uint8(2 << 2 * q)  # code 32
    b = b.reshape(-1)
    dense = K.np_dequant(ty, rows, cols, b)
    assert not dense[~keep].any()
    return b


@pytest.mark.parametrize("ty", QUANTIZED, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("large", [1, 7, 8, 20])
def test_small_activations_beside_large_ones_of_zero_weights(gpu, ty, large):
    """The sum is the small ones' alone: they must not be held to what the large ones allow, down to 2^-40 of them."""
    rng = np.random.default_rng(23 + 8 * ty + large)
    rows, tokens = 33, 56
    for cols, top in ((K.QK[ty], 0), (512, 0), (512, -61)):
        x = np.zeros((tokens, cols), np.float32)
        keep = np.zeros(cols, bool)
        for g in range(cols // 32):
            at = 32 * g + rng.permutation(32)[:large + 5]
            x[:, at[:large]] = rng.uniform(0.5, 1, (tokens, large)) * 2.0 ** top
            keep[at[large:]] = True
            for t in range(tokens):  # one to five of them, 2^-13 .. 2^-40 below the large ones
                n = 1 + t % 5
                x[t, at[large:large + n]] = rng.choice([-1, 1], n) * rng.uniform(0.5, 1, n) * 2.0 ** (top - 13 - t % 28)
        w = _keep_columns(ty, rows, cols, K.random_packed(ty, rows, cols, rng), np.broadcast_to(keep, (rows, cols)))
        y = _product(gpu, ty, rows, cols, x, w)
        exact, mag = O.gemm_f64_mag(ty, cols, tokens, w, x.reshape(-1), rows)
        assert np.all(np.abs(y.astype(np.float64) - exact) <= K.single_kernel_bound(32, mag))


def _spread(kind, rng, shape):
    n = rng.normal(0, 1, shape)
    if kind == "swiglu":
        n = 3 * n / (1 + np.exp(-3 * n)) * 3 * rng.normal(0, 1, shape)
    elif kind == "lognormal":
        n = n * np.exp(2 * rng.normal(0, 1, shape))
    elif kind == "outliers":
        n[:, 5::97] *= 1e4
    return n.astype(np.float32)


@pytest.mark.parametrize("ty", QUANTIZED, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("kind", ["normal", "swiglu", "lognormal", "outliers"])
def test_rows_of_one_weight(gpu, ty, kind):
    """One product per result: three exact parts, two additions and the weight's scale, a rounding each."""
    rng = np.random.default_rng(61 + ty)
    rows, cols, tokens = 512, 512, 100
    x = _spread(kind, rng, (tokens, cols))
    w = _keep_columns(ty, rows, cols, K.random_packed(ty, rows, cols, rng), np.eye(cols, dtype=bool)[rng.permutation(cols)])
    y = _product(gpu, ty, rows, cols, x, w)
    exact, mag = O.gemm_f64_mag(ty, cols, tokens, w, x.reshape(-1), rows)
    assert np.all(np.abs(y.astype(np.float64) - exact) <= 8 * K.U * np.asarray(mag) + 2.0 ** -120)


@pytest.mark.parametrize("ty", QUANTIZED, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("tokens", [33, 70])
def test_chain_of_activations_of_wide_range(pkg, gpu, ty, tokens):
    """Rows that the sums' launches leave cut for the next product (add + RMSNorm, SiLU(gate) * up), with outliers in them:
    the product reads what it reads when the same rows are given to it plain."""
    hip = importlib.import_module("llama-rust_amd.hiprt")
    rng = np.random.default_rng(400 + ty + tokens)
    d, ff = 512, 768
    m_o, m_g, m_u = (gpu.upload_packed(ty, r, d, K.random_packed(ty, r, d, rng)) for r in (d, ff, ff))
    w_d = K.random_packed(ty, d, ff, rng)
    m_d = gpu.upload_packed(ty, d, ff, w_d)
    dev = lambda a: hip.DeviceBuffer.from_numpy(np.ascontiguousarray(a, np.float32).reshape(-1))
    x0, res = _spread("lognormal", rng, (tokens, d)), _spread("lognormal", rng, (tokens, d)) * np.float32(1e-3)
    res[::3, 7::50] = 3e4
    d_xn, d_gate, d_up, d_y = (hip.DeviceBuffer(tokens * n * 4) for n in (d, ff, ff, d))
    d_x0, d_res, d_norm = dev(x0), dev(res), dev(np.ones(d))
    a_o, a_gu, a_d = gpu.act_create(ty, d, tokens), gpu.act_create(ty, d, tokens), gpu.act_create(ty, ff, tokens)
    gpu.act_split_device(a_o, tokens, d_x0.ptr)
    gpu.gemm_act_device([m_o], a_o, tokens, None, pkg.EPILOGUE_ADD_RMSNORM, d_res.ptr, d_norm.ptr, 1e-5, d_xn.ptr, a_gu)
    gpu.gemm_act_device([m_g, m_u], a_gu, tokens, [d_gate.ptr, d_up.ptr])
    gpu.gemm_act_device([m_g, m_u], a_gu, tokens, None, pkg.EPILOGUE_SWIGLU, next_act=a_d)
    gpu.gemm_act_device([m_d], a_d, tokens, [d_y.ptr])
    gpu.synchronize()
    xn, gate, up = (b.to_numpy(np.float32).reshape(tokens, n) for b, n in ((d_xn, d), (d_gate, ff), (d_up, ff)))

    def product(m, rows, x):
        y = np.full(tokens * rows, np.nan, np.float32)
        gpu.gemm_resident(m, tokens, x.reshape(-1), y)
        return y.reshape(tokens, rows)

    assert np.array_equal(gate, product(m_g, ff, xn)) and np.array_equal(up, product(m_u, ff, xn))
    g64 = gate.astype(np.float64)
    with np.errstate(over="ignore"):
        h = (g64 / (1 + np.exp(-g64)) * up).astype(np.float32)
    exact, mag = O.gemm_f64_mag(ty, ff, tokens, w_d, h.reshape(-1), d)
    # SiLU(gate) * up is formed with another exp, good to 16 roundings
    assert np.all(np.abs(d_y.to_numpy(np.float32).reshape(tokens, d) - exact) <= (K.observed_envelope_u(ff) + 16) * K.U * np.asarray(mag) + 1e-30)


@pytest.mark.parametrize("ty", QUANTIZED, ids=lambda t: O.TYPE_NAMES[t])
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

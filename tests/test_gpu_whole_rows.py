"""Products whose workgroups own whole rows (gemm_whole_kernel, csrc/gemm_kernels.inc), against the oracle's float64
product.

Tolerances as in test_gpu_parity.py: the proven bound of any f32 summation order and the reference's observed envelope, both relative
to sum |w x| (langtax/src/simd/tests.rs:18-91)."""
import numpy as np
import pytest

import cases as K
import oracle as O

pytestmark = pytest.mark.gpu

QUANTIZED = [K.Q4_0, K.Q5_0, K.Q5_1, K.Q8_0, K.Q4_K, K.Q6_K]
# rows: edges of workgroups of 16, 32 and 64 rows and of the layout's 256; columns: fewer steps than wavefronts, shares of different length, an
# odd count of steps.  Which of them take whole rows, and how many wavefronts share them, is the plan's: test_gpu_whole_rows_variants.py has
# every variant, and asks the plan.
SHAPES = [(1, 32), (15, 96), (17, 480), (255, 1056), (300, 2080), (4096, 96), (4097, 288), (4130, 2304), (8193, 160), (8255, 2048), (16385, 96)]


@pytest.fixture(scope="module")
def gpu(pkg):
    g = pkg.HipGemv(0)
    yield g
    g.close()


def _check(ty, rows, cols, x, w, y):
    exact, mag = O.gemm_f64_mag(ty, cols, x.shape[0], w, x.reshape(-1), rows)
    err = np.abs(y.reshape(exact.shape).astype(np.float64) - exact)
    assert np.all(np.isfinite(y))
    assert np.all(err <= K.single_kernel_bound(cols, mag))
    assert np.all(err <= K.observed_envelope_u(cols) * K.U * mag)


@pytest.mark.parametrize("ty", QUANTIZED, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_edges(gpu, ty, rows, cols):
    cols = (cols + K.QK[ty] - 1) // K.QK[ty] * K.QK[ty]
    rng = np.random.default_rng(3 * rows + cols + ty)
    w = K.random_packed(ty, rows, cols, rng)
    m = gpu.upload_packed(ty, rows, cols, w)
    for tokens in (3, 8, 9, 16):
        x = rng.normal(0, 1, (tokens, cols)).astype(np.float32)
        x[0, ::7] *= 3.0e4
        y = np.full(tokens * rows, np.nan, np.float32)
        gpu.gemm_resident(m, tokens, x.reshape(-1), y)
        _check(ty, rows, cols, x, w, y)
    m.close()


@pytest.mark.parametrize("ty", QUANTIZED, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("rows,cols", [(1, 32), (300, 2080), (4097, 288), (8255, 160)])
def test_token_tiles(gpu, ty, rows, cols):
    """More tokens than a tile has slots: last tiles of one token, of all but one, and whole ones."""
    cols = (cols + K.QK[ty] - 1) // K.QK[ty] * K.QK[ty]
    rng = np.random.default_rng(5 * rows + cols + ty)
    w = K.random_packed(ty, rows, cols, rng)
    m = gpu.upload_packed(ty, rows, cols, w)
    for tokens in (9, 17, 31, 64, 65):
        x = rng.normal(0, 1, (tokens, cols)).astype(np.float32)
        x[-1, ::7] *= 3.0e4
        y = np.full(tokens * rows, np.nan, np.float32)
        gpu.gemm_resident(m, tokens, x.reshape(-1), y)
        _check(ty, rows, cols, x, w, y)
    m.close()


@pytest.mark.parametrize("ty", QUANTIZED, ids=lambda t: O.TYPE_NAMES[t])
def test_matrices_of_one_launch(gpu, ty):
    """Products of different rows and tokens that share a launch, and the same one after the other: the same workgroups' work."""
    rng = np.random.default_rng(40 + ty)
    cols, rows, tokens = 1024, [33, 256, 1, 100], [3, 8, 5, 4]
    ws = [K.random_packed(ty, r, cols, rng) for r in rows]
    ms = [gpu.upload_packed(ty, r, cols, w) for r, w in zip(rows, ws)]
    xs = [rng.normal(0, 1, (t, cols)).astype(np.float32) for t in tokens]
    ys = np.full(sum(r * t for r, t in zip(rows, tokens)), np.nan, np.float32)
    gpu.gemm_grouped(ms, tokens, np.concatenate([x.reshape(-1) for x in xs]), ys)
    at = 0
    for r, t, w, x in zip(rows, tokens, ws, xs):
        _check(ty, r, cols, x, w, ys[at:at + r * t])
        at += r * t
    for m in ms:
        m.close()


@pytest.mark.parametrize("ty", QUANTIZED, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("shift", [0, 4 * 1024])
def test_results_over_the_input(pkg, gpu, ty, shift):
    """y in x's place, and reaching into it: more than 32 tokens of a square matrix, whose activations are cut before anything is stored."""
    import importlib
    hip = importlib.import_module("llama-rust_amd.hiprt")
    n = 1024
    rng = np.random.default_rng(70 + ty)
    w = K.random_packed(ty, n, n, rng)
    m = gpu.upload_packed(ty, n, n, w)
    for tokens in (33, 64):
        x = rng.normal(0, 1, (tokens, n)).astype(np.float32)
        both = np.zeros(tokens * n + shift, np.float32)
        both[shift:] = x.reshape(-1)
        buf = hip.DeviceBuffer.from_numpy(both)
        gpu.gemm_device(m, tokens, buf.ptr + 4 * shift, buf.ptr)
        gpu.synchronize()
        _check(ty, n, n, x, w, buf.to_numpy(np.float32)[:tokens * n])
        buf.free()
    m.close()

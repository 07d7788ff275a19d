"""Every variant of gemm_whole_kernel (csrc/gemm_kernels.inc) that the plan picks, against the oracle's float64 product, and its activations
cut beforehand or normed as they are read against plain ones, bit for bit.

Tolerances as in test_gpu_whole_rows.py."""
import importlib
import os
import subprocess
import sys

import numpy as np
import pytest

import cases as K
import oracle as O
import whole_rows as W
from test_gpu_whole_rows import _check

pytestmark = pytest.mark.gpu

QUANTIZED = W.BLOCKS + [K.Q4_K, K.Q6_K]


@pytest.fixture(scope="module")
def gpu(pkg):
    g = pkg.HipGemv(0)
    yield g
    g.close()


@pytest.mark.parametrize("ty,product", [(ty, p) for ty in QUANTIZED for p in W.VARIANTS[ty]],
                         ids=lambda v: O.TYPE_NAMES[v] if isinstance(v, int) else "x".join(map(str, v)))
def test_variant(lib, gpu, ty, product):
    rows, cols, tokens, wg_rows, waves = product
    assert W.planned(lib, ty, [rows], cols, tokens) == (wg_rows, waves)
    rng = np.random.default_rng(rows + cols + 100 * tokens + ty)
    w = K.random_packed(ty, rows, cols, rng)
    m = gpu.upload_packed(ty, rows, cols, w)
    x = rng.normal(0, 1, (tokens, cols)).astype(np.float32)
    x[-1, ::7] *= 3.0e4
    y = np.full(tokens * rows, np.nan, np.float32)
    gpu.gemm_resident(m, tokens, x.reshape(-1), y)
    _check(ty, rows, cols, x, w, y)
    m.close()


@pytest.mark.parametrize("ty,product", [(ty, p) for ty in QUANTIZED for p in W.CHAINED[ty]],
                         ids=lambda v: O.TYPE_NAMES[v] if isinstance(v, int) else "x".join(map(str, v)))
def test_cut_and_normed_activations(lib, pkg, gpu, ty, product):
    """A product of a chain, of activations an epilogue has cut and (up to 32 tokens) of rows whose norm it left to the product, alone and with
    the residual epilogue: the bits of the plain product of the same rows."""
    rows, cols, tokens, wg_rows, waves = product
    assert W.planned(lib, ty, [rows], cols, tokens) == (wg_rows, waves)
    hip = importlib.import_module("llama-rust_amd.hiprt")
    rng = np.random.default_rng(rows + cols + 100 * tokens + ty)
    w = K.random_packed(ty, rows, cols, rng, signed=False, scale=0.05)
    m = gpu.upload_packed(ty, rows, cols, w)
    m_o = gpu.upload_packed(ty, cols, 256, K.random_packed(ty, cols, 256, rng, signed=False, scale=0.05))
    x0, res0 = rng.normal(0, 1, (tokens, 256)), rng.normal(0, 1, (tokens, cols))
    res1 = rng.normal(0, 1, (tokens, rows)).astype(np.float32)
    dev = lambda a: hip.DeviceBuffer.from_numpy(np.ascontiguousarray(a, np.float32).reshape(-1))
    d_x0, d_g, d_g1 = dev(x0), dev(1 + rng.normal(0, 0.05, cols)), dev(np.ones(rows))
    d_xn, d_y = hip.DeviceBuffer(4 * tokens * cols), [hip.DeviceBuffer(4 * tokens * rows) for _ in range(3)]
    a_cut, a_norm, a_next = gpu.act_create(ty, cols, tokens), gpu.act_create(ty, cols, tokens), gpu.act_create(ty, rows, tokens)
    bits = lambda b: b.to_numpy(np.float32).view(np.uint32)
    d_res = [dev(res0), dev(res0)]
    gpu.gemm_plain_act_device([m_o], d_x0.ptr, tokens, None, pkg.EPILOGUE_ADD_RMSNORM, d_res[0].ptr, d_g.ptr, 1e-5, d_xn.ptr, a_cut)
    gpu.gemm_device(m, tokens, d_xn.ptr, d_y[0].ptr)
    acts = [a_cut]
    if tokens <= 32:
        gpu.gemm_plain_act_device([m_o], d_x0.ptr, tokens, None, pkg.EPILOGUE_ADD_RMSNORM_DEFERRED, d_res[1].ptr, d_g.ptr, 1e-5, 0, a_norm)
        acts.append(a_norm)
    gpu.synchronize()
    xn, y = d_xn.to_numpy(np.float32).reshape(tokens, cols), d_y[0].to_numpy(np.float32)
    _check(ty, rows, cols, xn, w, y)
    for a, d in zip(acts, d_y[1:]):
        gpu.gemm_act_device([m], a, tokens, [d.ptr])
        gpu.synchronize()
        assert np.array_equal(bits(d), y.view(np.uint32))
        d_sum = dev(res1)
        if tokens <= 32:
            gpu.gemm_act_device([m], a, tokens, None, pkg.EPILOGUE_ADD_RMSNORM_DEFERRED, d_sum.ptr, d_g1.ptr, 1e-5, 0, a_next)
        else:
            gpu.gemm_act_device([m], a, tokens, None, pkg.EPILOGUE_ADD_RMSNORM, d_sum.ptr, d_g1.ptr, 1e-5, 0, a_next)
        gpu.synchronize()
        assert np.array_equal(bits(d_sum), (res1 + y.reshape(tokens, rows)).reshape(-1).view(np.uint32))
        d_sum.free()
    for a in (a_cut, a_norm, a_next):
        a.close()
    for b in d_y + d_res + [d_x0, d_g, d_g1, d_xn]:
        b.free()
    m.close()
    m_o.close()


@pytest.mark.parametrize("ty", QUANTIZED, ids=lambda t: O.TYPE_NAMES[t])
def test_products_of_several_token_tiles_in_one_launch(lib, gpu, ty):
    """Products of different rows and counts of token tiles that share a launch, and each in a launch of its own: the same bits, as their
    wavefronts depend on the columns alone."""
    rng = np.random.default_rng(90 + ty)
    cols, rows, tokens = 512, [33, 200, 65, 16], [17, 65, 33, 18]
    for some in ([0], [1], [2], [3], [0, 1, 2, 3]):
        assert W.planned(lib, ty, [rows[i] for i in some], cols, [tokens[i] for i in some])[0] != 0
    ws = [K.random_packed(ty, r, cols, rng) for r in rows]
    ms = [gpu.upload_packed(ty, r, cols, w) for r, w in zip(rows, ws)]
    xs = [rng.normal(0, 1, (t, cols)).astype(np.float32) for t in tokens]
    ys = np.full(sum(r * t for r, t in zip(rows, tokens)), np.nan, np.float32)
    gpu.gemm_grouped(ms, tokens, np.concatenate([x.reshape(-1) for x in xs]), ys)
    at = 0
    for r, t, w, m, x in zip(rows, tokens, ws, ms, xs):
        y = np.full(t * r, np.nan, np.float32)
        gpu.gemm_resident(m, t, x.reshape(-1), y)
        assert np.array_equal(ys[at:at + r * t].view(np.uint32), y.view(np.uint32))
        _check(ty, r, cols, x, w, y)
        at += r * t
        m.close()


FIRST_LAUNCH_IS_RECORDED = r"""
import importlib, sys
import numpy as np
sys.path[:0] = [{root!r}, {root!r} + "/tests"]
import cases as K
import whole_rows as W
pkg = importlib.import_module("llama-rust_amd")
hip = importlib.import_module("llama-rust_amd.hiprt")
gpu, rng = pkg.HipGemv(0), np.random.default_rng(7)
rows, cols, tokens = 512, 2048, 8
assert W.planned(pkg.load_library(), K.Q4_0, [rows], cols, tokens) == (16, 16)  # sixteen wavefronts: more than 48 KB of LDS
m, larger = (gpu.upload_packed(ty, r, cols, K.random_packed(ty, r, cols, rng)) for ty, r in ((K.Q4_0, rows), (K.Q8_0, 4 * rows)))
gpu.prepare(m, tokens)
x = hip.DeviceBuffer.from_numpy(rng.normal(0, 1, tokens * cols).astype(np.float32))
y, y2 = hip.DeviceBuffer(4 * tokens * rows), hip.DeviceBuffer(16 * tokens * rows)
gpu.gemm_device(larger, tokens, x.ptr, y2.ptr)  # the workspace, by another dtype's kernel
gpu.synchronize()
stream = hip.Stream()
graph = hip.Graph(stream, lambda s: gpu.gemm_device(m, tokens, x.ptr, y.ptr, s.ptr))
gpu.gemm_device(m, tokens, x.ptr, y2.ptr)
gpu.synchronize()
want = y2.to_numpy(np.float32, tokens * rows)
assert np.all(np.isfinite(want)) and np.any(want)
for replay in range(3):
    y.fill_byte(255)
    hip.device_synchronize()
    graph.launch()
    stream.synchronize()
    assert np.array_equal(y.to_numpy(np.float32), want), replay
graph.destroy()
print("recorded")
"""


def test_first_launch_inside_a_capture():
    """In a process of its own: the kernel's LDS limit is raised at its first launch, which a stream under capture records."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    done = subprocess.run([sys.executable, "-c", FIRST_LAUNCH_IS_RECORDED.format(root=root)], capture_output=True, text=True, timeout=100)
    assert done.returncode == 0 and done.stdout.strip().endswith("recorded"), done.stdout + done.stderr

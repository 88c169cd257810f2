"""GPU parity of the wide batched GEMM (hip_gemm, hip_gemm_grouped[_ex] at prompt
sizes) on Q4_K, Q5_K, Q6_K, IQ3_S and IQ2_XXS, against float64 sums of the
closed-form weights on a sample of rows (both ends, tile edges, the middle).

Bound: x is kept to at least 21 bits per element (relative 2^-21), so an
output's error is at most 2^-21 sum |w x| plus f32 rounding of the sums; the
2-norm over the sampled outputs is held to 2^-20 of that sum's norm, with a
format's scaled quant and its minimum counted apart.
"""
import numpy as np
import pytest

import closed_form as cf
from saient_quartz_amd import GGML_TYPES, synth, type_size
from saient_quartz_amd.api import check
from saient_quartz_amd.host import GpuBuf, gemm_grouped_async, gemm_grouped_ex_async

pytestmark = pytest.mark.gpu


def sample(out_dim):
    rows = set(range(0, 34)) | set(range(out_dim - 34, out_dim))
    for edge in (256, out_dim // 2):
        rows |= set(range(edge - 2, edge + 2))
    return np.array(sorted(r for r in rows if 0 <= r < out_dim))


def reference(t, x, data, in_dim, rows):
    """-> (float64 products, float64 sums of magnitudes) of the sampled rows."""
    size = type_size(t, in_dim)
    d = data.reshape(-1, size)[rows].reshape(-1)
    w = cf.decode(t, d).astype(np.float64).reshape(len(rows), in_dim)
    mag = np.abs(w)
    if t in (12, 13):  # |d sc q| <= |w| + |dmin m|
        b = d.reshape(-1, GGML_TYPES[t][2]).astype(np.int64)
        m = cf.f16(b[:, 2], b[:, 3])[:, None] * cf.k4_scales(b[:, 4:16])[1]
        mag = mag + 2 * np.abs(np.repeat(m, 32, axis=1).reshape(len(rows), in_dim))
    x = x.astype(np.float64)
    return x @ w.T, np.abs(x) @ mag.T


def held(got, ref, mag):
    err = np.linalg.norm(got - ref, axis=1) / np.linalg.norm(mag, axis=1)
    assert err.max() < 2.0**-20, err.max()


# 64-token tiles (odd tokens, a partial row tile, K split and not) and 128-token
# tiles; 9 groups of 256
@pytest.mark.parametrize("t", [12, 13, 14, 21, 16])
@pytest.mark.parametrize("out_dim, in_dim, n", [(4100, 4096, 257), (9001, 2304, 301), (14400, 4096, 500)])
def test_wide_gemm(qh, t, out_dim, in_dim, n):
    data = synth.weights(t, out_dim, in_dim, seed=t + out_dim)
    x = synth.activations(n, in_dim, seed=n)
    x *= (10.0 ** np.linspace(-3, 3, n, dtype=np.float32))[:, None]  # every token has its own exponents
    x[:, ::97] *= 300.0  # outliers
    w, dx = GpuBuf.upload(data), GpuBuf.upload_f32(x.reshape(-1))
    dy = GpuBuf.upload_f32(np.full(n * out_dim + 1, 7.0))
    for _ in range(2):  # the second call finds the arrival counters at zero again
        check("hip_gemm", qh.hip_gemm(t, w.ptr, dx.ptr, dy.ptr, in_dim, out_dim, n))
        check("hip_sync", qh.hip_sync())
        y = dy.download(np.float32)
        assert y[-1] == 7.0
        rows = sample(out_dim)
        held(y[:-1].reshape(n, out_dim)[:, rows].astype(np.float64), *reference(t, x, data, in_dim, rows))


@pytest.mark.parametrize("t", [12, 14])
def test_wide_grouped(qh, t):
    """Matrices sharing x (its images written once), one of no rows between them
    and one with its own, shorter x behind them."""
    in_dim, outs, n = 4096, [4096, 0, 4200, 4100], [300, 400, 300, 260]
    data = [synth.weights(t, max(o, 1), in_dim, seed=30 + k) for k, o in enumerate(outs)]
    xs = [synth.activations(400, in_dim, seed=5), None, None, synth.activations(260, in_dim, seed=6)]
    w = [GpuBuf.upload(d) for d in data]
    dx = [GpuBuf.upload_f32(x.reshape(-1)) if x is not None else None for x in xs]
    dx[1] = dx[2] = dx[0]
    dy = [GpuBuf.alloc_f32(max(1, a * b)) for a, b in zip(n, outs)]
    gemm_grouped_async(qh, t, [b.ptr for b in w], [b.ptr for b in dx], [b.ptr for b in dy], n, outs, in_dim, None)
    check("hip_sync", qh.hip_sync())
    for k in (0, 2, 3):
        rows = sample(outs[k])
        x = (xs[0] if k < 3 else xs[3])[:n[k]]
        got = dy[k].download(np.float32)[:n[k] * outs[k]].reshape(n[k], outs[k])[:, rows]
        held(got.astype(np.float64), *reference(t, x, data[k], in_dim, rows))


@pytest.mark.parametrize("t", [14, 21])
def test_wide_swiglu_residual(qh, t):
    """y += W (silu(gate) * up) at prompt size, and a token holding an infinity."""
    in_dim, out_dim, n = 14336, 4096, 130
    data = synth.weights(t, out_dim, in_dim, seed=t)
    gate, up = synth.activations(n, in_dim, seed=1), synth.activations(n, in_dim, seed=2)
    y0 = synth.activations(n, out_dim, seed=3)
    gate[7, 1000] = np.inf
    w, dg, du = GpuBuf.upload(data), GpuBuf.upload_f32(gate.reshape(-1)), GpuBuf.upload_f32(up.reshape(-1))
    dy = GpuBuf.upload_f32(y0.reshape(-1))
    gemm_grouped_ex_async(qh, t, [w.ptr], [dg.ptr], [dy.ptr], [n], [out_dim], in_dim, None, up_ptrs=[du.ptr],
                          accumulate=True)
    check("hip_sync", qh.hip_sync())
    got = dy.download(np.float32).reshape(n, out_dim)
    assert not np.isfinite(got[7]).any()
    ok = np.arange(n) != 7
    g = gate[ok].astype(np.float64)
    rows = sample(out_dim)
    ref, mag = reference(t, (g / (1 + np.exp(-g)) * up[ok]), data, in_dim, rows)
    held(got[ok][:, rows].astype(np.float64), ref + y0[ok][:, rows], mag + np.abs(y0[ok][:, rows]))

"""GPU parity of the batched GEMM of 5 .. 16 tokens on few rows (hip_gemm,
hip_gemm_grouped[_ex]) on Q4_K, Q5_K and Q6_K: one workgroup per 32 rows, whole K.
Reference and bound as for the wide kernel's test.
"""
import numpy as np
import pytest

from saient_quartz_amd import synth
from saient_quartz_amd.api import check
from saient_quartz_amd.host import GpuBuf, gemm_grouped_ex_async
from test_gpu_mmw import held, reference, sample

pytestmark = pytest.mark.gpu


def tokens(n, in_dim, seed):
    x = synth.activations(n, in_dim, seed=seed)
    x *= (10.0 ** np.linspace(-3, 3, n, dtype=np.float32))[:, None]  # every token has its own exponents
    x[:, ::97] *= 300.0
    return x


# fewer groups of 256 than wavefronts, one more than them, a row, a partial tile, the
# last one-round size and the first beyond it
@pytest.mark.parametrize("t", [12, 13, 14])
@pytest.mark.parametrize("out_dim, in_dim, n", [(1, 256, 16), (33, 512, 9), (95, 2304, 13), (2050, 2048, 5), (4096, 4096, 16),
                                                (8192, 2048, 11), (8193, 2048, 11)])
def test_few_rows_gemm(qh, t, out_dim, in_dim, n):
    data = synth.weights(t, out_dim, in_dim, seed=t + out_dim)
    x = tokens(n, in_dim, n)
    w, dx = GpuBuf.upload(data), GpuBuf.upload_f32(x.reshape(-1))
    dy = GpuBuf.upload_f32(np.full(n * out_dim + 1, 7.0))
    check("hip_gemm", qh.hip_gemm(t, w.ptr, dx.ptr, dy.ptr, in_dim, out_dim, n))
    check("hip_sync", qh.hip_sync())
    y = dy.download(np.float32)
    assert y[-1] == 7.0
    rows = sample(out_dim)
    held(y[:-1].reshape(n, out_dim)[:, rows].astype(np.float64), *reference(t, x, data, in_dim, rows))


@pytest.mark.parametrize("t", [12, 14])
def test_few_rows_grouped_swiglu_residual(qh, t):
    """Matrices of different heights sharing x (one of no rows), y += W (silu(gate) *
    up), and a token holding an infinity."""
    in_dim, outs, n = 2048, [300, 0, 40, 1024], 13
    data = [synth.weights(t, max(o, 1), in_dim, seed=k) for k, o in enumerate(outs)]
    gate, up = synth.activations(n, in_dim, seed=1), synth.activations(n, in_dim, seed=2)
    gate[7, 1000] = np.inf
    y0 = [synth.activations(n, max(o, 1), seed=9 + k) for k, o in enumerate(outs)]
    w, dg, du = [GpuBuf.upload(d) for d in data], GpuBuf.upload_f32(gate.reshape(-1)), GpuBuf.upload_f32(up.reshape(-1))
    dy = [GpuBuf.upload_f32(y.reshape(-1)) for y in y0]
    gemm_grouped_ex_async(qh, t, [b.ptr for b in w], [dg.ptr] * 4, [b.ptr for b in dy], [n] * 4, outs, in_dim, None,
                          up_ptrs=[du.ptr] * 4, accumulate=True)
    check("hip_sync", qh.hip_sync())
    ok = np.arange(n) != 7
    g = gate[ok].astype(np.float64)
    for k, o in enumerate(outs):
        if not o:
            continue
        got = dy[k].download(np.float32).reshape(n, o)
        assert not np.isfinite(got[7]).any()
        rows = sample(o)
        ref, mag = reference(t, g / (1 + np.exp(-g)) * up[ok], data[k], in_dim, rows)
        y = y0[k][ok][:, rows]
        held(got[ok][:, rows].astype(np.float64), ref + y, mag + np.abs(y))

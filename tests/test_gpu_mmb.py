"""GPU parity of the batched block-format GEMM (hip_gemm on Q4_0, Q4_1, Q5_0, Q5_1,
Q8_0 and IQ4_NL with n >= 2) against float64 sums of the closed-form weights.

Bound: x is kept to 21 bits per element (relative 2^-21, truncated), so the
error of an output is at most 2^-21 sum |w x| from x plus f32 rounding of the
sums; the 2-norm over a token's outputs is held to 2^-20 of that sum's norm,
where w counts a format's scaled quant and its minimum apart.
"""
import numpy as np
import pytest

import closed_form as cf
from saient_quartz_amd import GGML_TYPES, synth
from saient_quartz_amd.api import check
from saient_quartz_amd.host import GpuBuf

pytestmark = pytest.mark.gpu

BLOCK_TYPES = [2, 3, 6, 7, 8, 20]


def gemm(qh, t, x, data, in_dim, out_dim, n):
    w, dx = GpuBuf.upload(data), GpuBuf.upload_f32(x.reshape(-1))
    dy = GpuBuf.upload_f32(np.full(n * out_dim + 1, 7.0))
    check("hip_gemm", qh.hip_gemm(t, w.ptr, dx.ptr, dy.ptr, in_dim, out_dim, n))
    check("hip_sync", qh.hip_sync())
    y = dy.download(np.float32)
    assert y[-1] == 7.0
    return y[:-1].reshape(n, out_dim)


def magnitudes(t, data, out_dim, in_dim):
    w = np.abs(cf.decode(t, data).astype(np.float64)).reshape(out_dim, in_dim)
    if t in (3, 7):  # |scaled quant| + |minimum|
        b = data.reshape(-1, GGML_TYPES[t][2]).astype(np.int64)
        m = np.repeat(cf.f16(b[:, 2], b[:, 3]), 32).reshape(out_dim, in_dim)
        w = np.abs(cf.decode(t, data).astype(np.float64).reshape(out_dim, in_dim) - m) + np.abs(m)
    return w


# 16- and 32-row workgroups, row, token and K remainders, one block, a last group
# of fewer than 8 blocks (2880 = 11.25 groups), more tokens than one tile
@pytest.mark.parametrize("t", BLOCK_TYPES)
@pytest.mark.parametrize("out_dim, in_dim, n", [(37, 32, 3), (16, 256, 16), (33, 288, 17), (100, 2880, 5), (5, 4096, 31),
                                                (4100, 512, 40), (1, 1056, 64)])
def test_block_gemm(qh, t, out_dim, in_dim, n):
    data = synth.weights(t, out_dim, in_dim, seed=t + out_dim + in_dim)
    x = synth.activations(n, in_dim, seed=n + in_dim)
    x[:, ::97] *= 3000.0  # outliers
    got = gemm(qh, t, x, data, in_dim, out_dim, n).astype(np.float64)
    ref = cf.gemv_f64(t, x, data, in_dim, out_dim).T
    mag = np.abs(x).astype(np.float64) @ magnitudes(t, data, out_dim, in_dim).T
    err = np.linalg.norm(got - ref, axis=1) / np.linalg.norm(mag, axis=1)
    assert err.max() < 2.0**-20, err.max()


@pytest.mark.parametrize("t", [2, 6, 20])
def test_block_gemm_infinity(qh, t):
    """A token holding an infinity: +-Inf or NaN exactly where float64 gives them;
    the other tokens are untouched."""
    out_dim, in_dim, n = 64, 512, 4
    data = synth.weights(t, out_dim, in_dim, seed=t)
    x = synth.activations(n, in_dim, seed=3)
    ok = gemm(qh, t, x, data, in_dim, out_dim, n)
    x[1, 300], x[2, 5] = np.inf, np.nan
    got = gemm(qh, t, x, data, in_dim, out_dim, n)
    with np.errstate(invalid="ignore"):
        ref = cf.gemv_f64(t, x, data, in_dim, out_dim).T
    assert np.array_equal(got[1], ref[1].astype(np.float32), equal_nan=True)
    assert np.isnan(got[2]).all()
    assert np.array_equal(got[[0, 3]], ok[[0, 3]])

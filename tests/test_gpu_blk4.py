"""GPU parity of the matrix-core GEMV of Q4_0, Q5_0 and IQ4_NL (hip_gemv on 2^24 weights
and more) against float64 sums of the closed-form weights.

Bound: x keeps at least 24 bits (2^-25 of each element, or of 2^-6 of the largest |x|
near it), a piece's integer dot is rounded to f32 twice (2 x 2^-24) and the sums over
pieces are f32 sums of at most 2^7 terms per lane: below 2^-19 sum |w x| in all.
"""
import numpy as np
import pytest

import closed_form as cf
from saient_quartz_amd import synth, type_size
from saient_quartz_amd.api import check
from saient_quartz_amd.host import GpuBuf

pytestmark = pytest.mark.gpu


# rows that are and are not whole tiles of 11, 14 and 16; K in one chunk and in several,
# the last of one group; the first size below the kernel's range
@pytest.mark.parametrize("t", [2, 6, 20])
@pytest.mark.parametrize("out_dim, in_dim", [(4096, 4096), (4095, 4096), (4101, 4352), (2050, 8448), (1301, 14336)])
def test_block_gemv(qh, t, out_dim, in_dim):
    data = synth.weights(t, out_dim, in_dim, seed=t + out_dim)
    x = synth.activations(1, in_dim, seed=t).reshape(-1)
    x[::97] *= 300.0
    w, dx, dy = GpuBuf.upload(data), GpuBuf.upload_f32(x), GpuBuf.upload_f32(np.full(out_dim + 1, 7.0))
    check("hip_gemv", qh.hip_gemv(t, w.ptr, dx.ptr, dy.ptr, in_dim, out_dim))
    check("hip_sync", qh.hip_sync())
    y = dy.download(np.float32)
    assert y[-1] == 7.0
    rows = np.r_[0:40, out_dim // 2:out_dim // 2 + 40, out_dim - 40:out_dim]
    d = data.reshape(-1, type_size(t, in_dim))[rows].reshape(-1)
    wd = cf.decode(t, d).astype(np.float64).reshape(len(rows), in_dim)
    xd = x.astype(np.float64)
    assert (np.abs(y[rows] - wd @ xd) <= 2.0**-19 * (np.abs(wd) @ np.abs(xd))).all()
    # a token that is not finite
    x[77] = np.inf
    dx = GpuBuf.upload_f32(x)
    check("hip_gemv", qh.hip_gemv(t, w.ptr, dx.ptr, dy.ptr, in_dim, out_dim))
    check("hip_sync", qh.hip_sync())
    assert not np.isfinite(dy.download(np.float32)[:-1][wd_nonzero(data, t, in_dim, out_dim)]).any()


def wd_nonzero(data, t, in_dim, out_dim):
    """The rows whose weight 77 is not zero (the others may give 0 * Inf = NaN or skip it)."""
    rows = np.arange(0, out_dim, 501)
    d = data.reshape(-1, type_size(t, in_dim))[rows].reshape(-1)
    return rows[cf.decode(t, d).reshape(len(rows), in_dim)[:, 77] != 0]

"""Decode GEMV rows of one chunk column (K up to 2048: two row groups in flight) at
its edges, against the 64-bit product of the oracle's decoded weights.

K: a few chunks, one lane short of a column, a whole column, and the first lengths of
the two-column walk beyond it. Rows: fewer than a wave's, odd counts of row groups
(the pair's second half clamped), and more groups than stay resident, so that blocks
take several pairs.

Bar 4e-6 of the largest value (of the size of a sum with random signs where the few
values of a small case cancel below it): activations keep at least 22 bits, every sum
is f32, and over K <= 2304 products of random sign the error of the largest of 1e5
results stays below 2e-6."""
import numpy as np
import pytest

import oracle
import uaii_amd
from uaii_amd import synth, DeviceBuffer, DeviceWeight, check_hip

pytestmark = pytest.mark.gpu

TYPES = [uaii_amd.Q4_0, uaii_amd.Q4_1, uaii_amd.Q4_K, uaii_amd.Q5_K, uaii_amd.Q6_K]


def weights(t, rows, cols, seed):
    p = synth.quantize(t, synth.normals(seed, 1, 0, rows * cols, 0.02))
    return DeviceWeight(t, p, rows, cols), oracle.dequant(t, p, rows, cols).astype(np.float64)


@pytest.mark.parametrize("t", TYPES, ids=lambda t: uaii_amd.TYPE_NAMES[t])
@pytest.mark.parametrize("cols", [32, 256, 2016, 2048, 2080, 2304])
@pytest.mark.parametrize("rows", [1, 7, 33, 1000, 40000])
def test_gemv_one_column(hip, t, cols, rows):
    if t >= uaii_amd.Q2_K and cols % 256:
        pytest.skip("K-quant rows are whole super-blocks")
    if rows == 40000 and cols not in (256, 2048):
        pytest.skip("several pairs a block: at one short and one whole column")
    w, wf = weights(t, rows, cols, rows + cols + t)
    x = synth.normals(rows + cols, 2, 0, cols, 1.0)
    norm = 1 + synth.normals(rows + cols, 4, 0, cols, 0.2)
    y0 = synth.normals(rows + cols, 5, 0, rows, 1.0)
    dx, dn = DeviceBuffer.from_array(x), DeviceBuffer.from_array(norm)
    x64 = x.astype(np.float64)
    xn = x64 / np.sqrt((x64 ** 2).mean() + 1e-5) * norm
    typical = lambda v, m: float(np.sqrt((v ** 2) @ (m ** 2).T).max())

    def close(dy, want, floor):
        got = dy.to_array(np.float32, rows)
        err = np.abs(got - want).max() / max(np.abs(want).max(), floor)
        print(uaii_amd.TYPE_NAMES[t], rows, cols, "maxrel %.2e" % err, flush=True)
        assert err < 4e-6

    dy = DeviceBuffer.from_array(y0)
    check_hip(hip.uaii_hip_gemv(w.h, dx.ptr, dy.ptr, None))
    check_hip(hip.uaii_hip_synchronize())
    close(dy, x64 @ wf.T, typical(x64, wf))
    dy = DeviceBuffer.from_array(y0)
    check_hip(hip.uaii_hip_gemv_add(w.h, dx.ptr, None, 0.0, dy.ptr, None))
    check_hip(hip.uaii_hip_synchronize())
    close(dy, y0 + x64 @ wf.T, typical(x64, wf))
    if rows < 40000:
        u, uf = weights(t, rows, cols, rows + cols + t + 1)
        check_hip(hip.uaii_hip_gemv_swiglu(w.h, u.h, dx.ptr, dn.ptr, 1e-5, dy.ptr, None))
        check_hip(hip.uaii_hip_synchronize())
        g = xn @ wf.T
        close(dy, g / (1 + np.exp(-g)) * (xn @ uf.T), 0.5 * typical(xn, wf) * typical(xn, uf))

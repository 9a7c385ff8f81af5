"""The row GEMM (k_pf_mm) at the edges of its tiles, splits and formats, against the
64-bit product of the oracle's decoded weights.

Bar 4e-6 (maximum difference over the largest value, or over the size that sums of
such terms with random signs have where the few values of a small case happen to
cancel below it): the activations keep at least
22 bits (2^-23 of an element) and every sum is f32; over K <= 4096 products of
random sign the sums' error is below 3e-7 of the result's root mean square (measured
1e-7 .. 2.2e-7 over K = 2048 .. 14336), and the largest of up to 1e5 such errors is
below six times that."""
import numpy as np
import pytest

import oracle
import uaii_amd
from uaii_amd import synth, DeviceBuffer, DeviceWeight, check_hip

pytestmark = pytest.mark.gpu

TYPES = [uaii_amd.Q4_0, uaii_amd.Q8_0, uaii_amd.F16, uaii_amd.Q4_K, uaii_amd.Q5_K, uaii_amd.Q6_K]


def weights(t, rows, cols, seed):
    p = synth.quantize(t, synth.normals(seed, 1, 0, rows * cols, 0.02))
    return DeviceWeight(t, p, rows, cols), oracle.dequant(t, p, rows, cols).astype(np.float64)


def check(hip, op, t, m, rows, cols):
    seed = m * 7 + rows + cols + t
    w, wf = weights(t, rows, cols, seed)
    x = synth.normals(seed, 2, 0, m * cols, 1.0).reshape(m, cols)
    x *= np.exp(synth.normals(seed, 3, 0, cols, 0.6))[None, :]  # channels of unlike size
    dx, norm = DeviceBuffer.from_array(x), 1 + synth.normals(seed, 4, 0, cols, 0.2)
    dn, x64 = DeviceBuffer.from_array(norm), x.astype(np.float64)
    y0 = synth.normals(seed, 5, 0, m * rows, 1.0).reshape(m, rows)
    dy = DeviceBuffer.from_array(y0)
    xn = x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + 1e-5) * norm
    size = lambda a, b: float(np.sqrt((a ** 2) @ (b ** 2).T).max())
    typical = size(x64 if op in ("plain", "add") else xn, wf)
    if op == "plain":
        check_hip(hip.uaii_hip_gemm(w.h, dx.ptr, m, dy.ptr, None))
        want = x64 @ wf.T
    elif op == "rmsnorm":
        check_hip(hip.uaii_hip_gemm_rmsnorm(w.h, dx.ptr, m, dn.ptr, 1e-5, dy.ptr, None))
        want = xn @ wf.T
    elif op == "add":
        check_hip(hip.uaii_hip_gemm_add(w.h, dx.ptr, m, None, 0.0, dy.ptr, None))
        want = y0 + x64 @ wf.T
    else:
        u, uf = weights(t, rows, cols, seed + 1)
        check_hip(hip.uaii_hip_gemm_swiglu(w.h, u.h, dx.ptr, m, dn.ptr, 1e-5, dy.ptr, None))
        g = xn @ wf.T
        want = g / (1 + np.exp(-g)) * (xn @ uf.T)
        typical *= 0.5 * size(xn, uf)  # silu(g) = g / 2 near 0
    check_hip(hip.uaii_hip_synchronize())
    got = dy.to_array(np.float32, m * rows).reshape(m, rows)
    err = float(np.abs(got - want).max() / max(np.abs(want).max(), typical))
    print(op, uaii_amd.TYPE_NAMES[t], m, rows, cols, "maxrel %.2e" % err, flush=True)
    assert err < 4e-6


# rows of activations at the 16-, 32- and 64-row blocks' edges; output columns at the
# 16-column subtile, the wave (32 and 64) and the block (128 and 256) edges
@pytest.mark.parametrize("t", TYPES, ids=lambda t: uaii_amd.TYPE_NAMES[t])
@pytest.mark.parametrize("m,rows", [(1, 1), (2, 15), (15, 16), (16, 17), (17, 63), (31, 64), (33, 65), (63, 127),
                                    (64, 129), (65, 255), (130, 257)])
def test_row_gemm_edges(hip, t, m, rows):
    for op in ("plain", "swiglu"):
        check(hip, op, t, m, rows, 512)


# K: one unit of 256 and its parts (formats of 32-value blocks), odd unit counts, and
# lengths that split over blocks and over a block's two wave groups
@pytest.mark.parametrize("t", TYPES, ids=lambda t: uaii_amd.TYPE_NAMES[t])
@pytest.mark.parametrize("cols", [64, 128, 192, 256, 320, 768, 1408, 2304, 4096])
def test_row_gemm_lengths(hip, t, cols):
    if t >= uaii_amd.Q2_K and cols % 256:
        pytest.skip("K-quant rows are whole super-blocks")
    for m, op in ((9, "add"), (20, "rmsnorm"), (100, "add")):
        check(hip, op, t, m, 200, cols)


# 64-row blocks: one and two wave groups, no split, and a launch of more than one round
@pytest.mark.parametrize("t", TYPES, ids=lambda t: uaii_amd.TYPE_NAMES[t])
@pytest.mark.parametrize("m,rows,cols,op", [(512, 4096, 768, "add"), (700, 3000, 512, "plain"),
                                            (1100, 4200, 512, "swiglu")])
def test_row_gemm_large(hip, t, m, rows, cols, op):
    check(hip, op, t, m, rows, cols)


# long rows: 16-, 32- and 64-row blocks on both sides of the lines in blocks times K, the
# 32-row ones with 32 rows and with a ragged 64, and K splits of unequal shares
@pytest.mark.parametrize("t", TYPES, ids=lambda t: uaii_amd.TYPE_NAMES[t])
@pytest.mark.parametrize("m,rows,cols,op", [(100, 1000, 8192, "plain"), (100, 1030, 8192, "add"),
                                            (17, 4100, 8192, "plain"), (65, 1000, 14336, "rmsnorm"),
                                            (100, 700, 14336, "swiglu"), (300, 500, 14336, "add"),
                                            (300, 1200, 512, "swiglu"), (500, 1408, 512, "swiglu")])
def test_row_gemm_row_tiles(hip, t, m, rows, cols, op):
    check(hip, op, t, m, rows, cols)


def test_row_gemm_unaligned_output(hip):
    """y on a 4-byte boundary and an odd row count: the fold's one-column form."""
    t, m, rows, cols = uaii_amd.Q4_0, 5, 333, 2048
    w, wf = weights(t, rows, cols, 3)
    x = synth.normals(3, 2, 0, m * cols, 1.0).reshape(m, cols)
    dx, dy = DeviceBuffer.from_array(x), DeviceBuffer(4 * m * rows + 4)
    y = uaii_amd.C.c_void_p(dy.ptr.value + 4)
    check_hip(hip.uaii_hip_gemm(w.h, dx.ptr, m, y, None))
    check_hip(hip.uaii_hip_synchronize())
    got = dy.to_array(np.float32, m * rows + 1)[1:].reshape(m, rows)
    want = x.astype(np.float64) @ wf.T
    assert np.abs(got - want).max() / np.abs(want).max() < 4e-6


@pytest.mark.parametrize("t", [uaii_amd.Q5_K, uaii_amd.Q8_0], ids=lambda t: uaii_amd.TYPE_NAMES[t])
def test_row_gemm_formats_agree_with_steps(hip, t):
    """The row path against the same rows taken one at a time (uaii_hip_gemv)."""
    m, rows, cols = 37, 300, 1024
    w, _ = weights(t, rows, cols, 9)
    x = synth.normals(9, 2, 0, m * cols, 1.0).reshape(m, cols)
    dx, dy, dz = DeviceBuffer.from_array(x), DeviceBuffer(4 * m * rows), DeviceBuffer(4 * m * rows)
    check_hip(hip.uaii_hip_gemm(w.h, dx.ptr, m, dy.ptr, None))
    for i in range(m):
        check_hip(hip.uaii_hip_gemv(w.h, uaii_amd.C.c_void_p(dx.ptr.value + 4 * i * cols),
                                    uaii_amd.C.c_void_p(dz.ptr.value + 4 * i * rows), None))
    check_hip(hip.uaii_hip_synchronize())
    got, want = dy.to_array(np.float32, m * rows), dz.to_array(np.float32, m * rows)
    assert np.abs(got - want).max() / np.abs(want).max() < 4e-6


def rows_and_steps(hip, w, x, rows):
    """The row product and the same rows one at a time."""
    m, cols = x.shape
    dx, dy, dz = DeviceBuffer.from_array(x), DeviceBuffer(4 * m * rows), DeviceBuffer(4 * m * rows)
    check_hip(hip.uaii_hip_gemm(w.h, dx.ptr, m, dy.ptr, None))
    for i in range(m):
        check_hip(hip.uaii_hip_gemv(w.h, uaii_amd.C.c_void_p(dx.ptr.value + 4 * i * cols),
                                    uaii_amd.C.c_void_p(dz.ptr.value + 4 * i * rows), None))
    check_hip(hip.uaii_hip_synchronize())
    return [b.to_array(np.float32, m * rows).reshape(m, rows) for b in (dy, dz)]


@pytest.mark.parametrize("scale", [0.02, 1e-6])  # 1e-6: subnormal f16 weights
@pytest.mark.parametrize("m,rows,cols", [(9, 256, 512), (9, 512, 4096), (100, 512, 2048), (300, 1024, 512)])
def test_f16_rows_keep_32_bits(hip, m, rows, cols, scale):
    """F16 rows (f32 operands) are as close to 64 bits as the per-row kernel: 0.72e-7 to
    0.91e-7 of the result against its 0.83e-7 to 0.98e-7."""
    wf = synth.normals(m + cols, 1, 0, rows * cols, scale).astype(np.float16)
    w = DeviceWeight(uaii_amd.F16, wf.view(np.uint8), rows, cols)
    x = synth.normals(m + cols, 2, 0, m * cols, 1.0).reshape(m, cols)
    x *= np.exp(synth.normals(m + cols, 3, 0, cols, 0.6))[None, :]
    got, steps = rows_and_steps(hip, w, x, rows)
    want = x.astype(np.float64) @ wf.reshape(rows, cols).astype(np.float64).T
    err = lambda a: float(np.linalg.norm(a - want) / np.linalg.norm(want))
    print(m, rows, cols, scale, "rows %.3e steps %.3e" % (err(got), err(steps)), flush=True)
    assert err(got) <= err(steps)


def test_f16_rows_infinities(hip):
    """Infinities and NaN in F16 weights and in activations, and finite values at the
    ends of f32: what each element is agrees with the per-row kernel's."""
    m, rows, cols = 20, 70, 256
    wf = synth.normals(4, 1, 0, rows * cols, 0.02).astype(np.float16).reshape(rows, cols)
    wf[3, 7], wf[5, 9], wf[6, 100], wf[8, :] = np.inf, -np.inf, np.nan, 0
    x = synth.normals(4, 2, 0, m * cols, 1.0).reshape(m, cols)
    x[2, 11], x[4, 250], x[5, 30], x[7, 7] = np.inf, -np.inf, np.nan, 0
    x[9] *= 1e37
    x[10] *= 1e-37
    got, want = rows_and_steps(hip, DeviceWeight(uaii_amd.F16, wf.view(np.uint8).reshape(-1), rows, cols), x, rows)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    assert np.array_equal(got[np.isinf(got)], want[np.isinf(want)])
    assert np.isinf(got[0, 3]) and np.isnan(got[7, 3]) and np.isinf(got[2, 0]) and np.isnan(got[2, 8])
    for i in range(m):  # each row at its own size
        ok = np.isfinite(want[i])
        if ok.any():
            assert np.abs(got[i][ok] - want[i][ok]).max() <= 4e-6 * np.abs(want[i][ok]).max(), i


@pytest.mark.parametrize("t", [t for t in TYPES if t != uaii_amd.F16], ids=lambda t: uaii_amd.TYPE_NAMES[t])
def test_row_gemm_extreme_rows(hip, t):
    """Rows of finite values near the largest and the smallest f32 holds, beside an
    ordinary one: each keeps its precision (the row's power-of-two scale)."""
    m, rows, cols = 5, 70, 512
    w, wf = weights(t, rows, cols, 21)
    x = synth.normals(21, 2, 0, m * cols, 1.0).reshape(m, cols)
    # |x| up to about 4 of each: past 2^115 and near 2^127; below 2^-100 and near 2^-126
    x *= np.float32([1, 2e35, 4e37, 1e-31, 1e-36])[:, None]
    dx, dy = DeviceBuffer.from_array(x), DeviceBuffer(4 * m * rows)
    check_hip(hip.uaii_hip_gemm(w.h, dx.ptr, m, dy.ptr, None))
    check_hip(hip.uaii_hip_synchronize())
    got, want = dy.to_array(np.float32, m * rows).reshape(m, rows), x.astype(np.float64) @ wf.T
    err = np.abs(got - want).max(1) / np.abs(want).max(1)
    print(uaii_amd.TYPE_NAMES[t], err, flush=True)
    assert (err < 4e-6).all()


def test_row_gemm_infinite_activation(hip):
    """An infinite activation of a Q8_0 product gives what it gives one row at a time."""
    m, rows, cols = 4, 70, 512
    w, wf = weights(uaii_amd.Q8_0, rows, cols, 22)
    x = synth.normals(22, 2, 0, m * cols, 1.0).reshape(m, cols)
    x[1, 100], x[2, 3] = np.inf, -np.inf
    got, want = rows_and_steps(hip, w, x, rows)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    assert np.array_equal(got[np.isinf(got)], want[np.isinf(want)]) and np.isinf(got[1]).sum() > rows // 2

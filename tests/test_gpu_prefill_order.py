"""Prompt attention (k_pf_attn) over its launch order and tile edges, against 64 bits.

The order numbers heads first, longest query tiles first, alternate bands reversed: the
cases have one band, a part of a second, several, and bands of one tile (as many kv
heads as CUs), for 4, 2, 1 and 3 query heads per kv head; every query is checked, so a
tile left out or taken twice shows. Keys end at and around the 64-key tile.

Bar 1e-5 of the largest value: K and V are exact in f16, queries and probabilities keep
22 bits and sums are f32; scores reach |s| < 20, whose f32 rounding (20 * 2^-24 and as
much again from log2 e) moves a probability by less than 5e-6 of itself."""
import numpy as np
import pytest

from uaii_amd import synth, DeviceBuffer, check_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkv,hd,p0,m", [
    (32, 8, 128, 0, 1), (32, 8, 128, 63, 16), (32, 8, 128, 48, 17), (32, 8, 64, 0, 513), (32, 8, 128, 5, 1040),
    (16, 8, 64, 64, 1100), (8, 8, 128, 1, 130), (6, 2, 64, 30, 65), (256, 256, 64, 3, 200)])
def test_prompt_attention_order(hip, nh, nkv, hd, p0, m):
    max_seq = p0 + m + 3
    q = synth.normals(m, 1, 0, m * nh * hd, 1.5).reshape(m, nh, hd)
    k, v = (synth.normals(m, i, 0, nkv * max_seq * hd, 1.0).reshape(nkv, max_seq, hd).astype(np.float16)
            for i in (2, 3))
    dq, dk, dv = (DeviceBuffer.from_array(x) for x in (q, k, v))
    dout = DeviceBuffer(4 * m * nh * hd)
    check_hip(hip.uaii_hip_attention_prefill(dq.ptr, dk.ptr, dv.ptr, max_seq, nh, nkv, hd, p0, m, dout.ptr, None))
    check_hip(hip.uaii_hip_synchronize())
    got = dout.to_array(np.float32, m * nh * hd).reshape(m, nh, hd)
    hidden = np.arange(p0 + m)[None, :] > p0 + np.arange(m)[:, None]
    worst = 0.0
    for h in range(nh):
        kk, vv = (x[h // (nh // nkv), :p0 + m].astype(np.float64) for x in (k, v))
        s = q[:, h].astype(np.float64) @ kk.T / np.sqrt(hd)
        s[hidden] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        want = p @ vv / p.sum(1, keepdims=True)
        worst = max(worst, float(np.abs(got[:, h] - want).max() / np.abs(want).max()))
    print(nh, nkv, hd, p0, m, "maxrel %.2e" % worst, flush=True)
    assert worst < 1e-5

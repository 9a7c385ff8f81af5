"""What sessions allocate and which path their prompts take, with the HIP runtime calls
answered on host memory (fake_hip.c) and kernels that do nothing. Each test is a child
process, whose libuaii_amd.so binds to the calls loaded before it."""
import subprocess
import sys
from pathlib import Path

import pytest

import uaii_amd
from uaii_amd import synth

HERE = Path(__file__).resolve().parent

DENSE = synth.ModelConfig(n_layers=2, dim=512, n_heads=8, n_kv_heads=2, ffn=1024, vocab=3000, ctx_len=512,
                          type_default=uaii_amd.Q4_K, seed=81)
OPEN = synth.ModelConfig(n_layers=2, dim=512, n_heads=8, n_kv_heads=2, ffn=1024, vocab=3000, ctx_len=0,
                         type_default=uaii_amd.Q4_0, seed=82)
MOE = synth.ModelConfig(n_layers=2, dim=512, n_heads=8, n_kv_heads=2, ffn=512, vocab=1200, ctx_len=512,
                        type_default=uaii_amd.Q4_0, n_experts=4, top_k=2, router_std=1.0 / 22, seed=83)

HEAD = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_capacity.argtypes, fake.fake_used.restype = [ctypes.c_size_t], ctypes.c_size_t
sys.path.insert(0, sys.argv[2])
import numpy as np
import uaii_amd
path = sys.argv[3]
def prompt(n): return np.arange(n, dtype=np.int64)
def rows(s): return "pf_attention" in s.profile_summary()
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so"
    header = Path("/opt/rocm/include")
    probe = so.parent / "cu.cpp"
    probe.write_text("#include <hip/hip_runtime_api.h>\n#include <cstdio>\n"
                     'int main() { std::printf("%d", (int)hipDeviceAttributeMultiprocessorCount); }\n')
    subprocess.run(["g++", "-D__HIP_PLATFORM_AMD__", "-I", str(header), "-o", str(so.parent / "cu"), str(probe)],
                   check=True)
    cu = subprocess.run([str(so.parent / "cu")], check=True, capture_output=True, text=True).stdout
    subprocess.run(["gcc", "-O1", "-w", "-shared", "-fPIC", "-DFAKE_CU_ATTRIBUTE=" + cu, "-o", str(so),
                    str(HERE / "fake_hip.c")], check=True)
    return so


def child(fake, path, body):
    r = subprocess.run([sys.executable, "-c", HEAD + body, str(fake), str(HERE.parent / "universal-ai-inference_amd"),
                        str(path)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


def test_prompt_buffers_give_way_to_a_larger_cache(fake):
    """With no byte budget, a cache that does not fit beside an f32 session's prompt
    buffers takes their place, and the prompt runs in token steps."""
    child(fake, synth.cached_model(OPEN), """
s = uaii_amd.Session(path, profile=True)
before = fake.fake_used()
s.generate(prompt(40), 2)
assert rows(s)
held = fake.fake_used() - before
cache = 2 * 2 * 128 * 4 * 4000  # layers, K and V, kv_dim, f32, positions
fake.fake_capacity(before + cache + (2 << 20) + held // 2)
s.generate(prompt(40), 3960)
assert fake.fake_used() <= before + cache + (2 << 20) + held // 2
""")


def test_prompt_buffers_give_way_to_the_sampler(fake):
    child(fake, synth.cached_model(DENSE), """
s = uaii_amd.Session(path)
s.set_device_sampler(True)
s.generate(prompt(40), 2)
fake.fake_capacity(fake.fake_used() + 4096)
s.generate_sampled(prompt(40), 4, uaii_amd.sample_params(temperature=0.8, top_k=5, seed=1))
""")


@pytest.mark.parametrize("f16", [False, True])
def test_moe_without_ffn_norm_takes_steps(fake, tmp_path, f16):
    """A MoE model without ffn_norm generates in token steps (the row routing needs the norm)."""
    data = Path(synth.cached_model(MOE)).read_bytes()
    assert data.count(b"ffn_norm.weight") == 2
    path = tmp_path / "bare.gguf"
    path.write_bytes(data.replace(b"ffn_norm.weight", b"ffn_none.weight"))
    child(fake, path, """
s = uaii_amd.Session(path, profile=True, kv_f16=%r)
s.generate(prompt(40), 2)
assert not rows(s) and not s.prefill_supported()
""" % f16)


def test_prefill_budget(fake):
    """The byte budget that lets an f16 session prefill 39 rows is no larger than what the
    buffers have always come to: per row the stream, QKV, query, attention and hidden rows,
    four splits of partials, hi + lo halves, one f32 a 32-block and a scale."""
    d, q, kv, ffn, m, mpad = 512, 512, 128, 1024, 39, 64
    budget = 4 * m * (d + (q + 2 * kv) + q + q + ffn) + 16 * m * (q + 2 * kv) + 4 * mpad * ffn + mpad * ffn // 8 + 4 * mpad
    child(fake, synth.cached_model(DENSE), """
def works(budget):
    try:
        s = uaii_amd.Session(path, budget_bytes=budget, kv_f16=True)
        if ask: s.generate(prompt(40), 2)
        s.close()
        return True
    except uaii_amd.UaiiError as e:
        assert "memory budget exceeded" in str(e), e
        return False
least = []
for ask in (False, True):
    lo, hi = 1, 1 << 28
    while hi - lo > 1:
        mid = (lo + hi) // 2
        if works(mid): hi = mid
        else: lo = mid
    least.append(hi)
print(least, least[1] - least[0])
assert least[1] - least[0] <= %d
""" % budget)

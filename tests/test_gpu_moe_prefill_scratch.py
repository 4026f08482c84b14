"""The scratch of a routed-expert prefill is sized for the prompt, and a
prefill whose scratch is refused serves its rows in batches of 16."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CFG = dict(n_layers=2, hidden=512, n_heads=4, n_kv=2, head_dim=128, inter=256, vocab=1024, max_seq=2200, rope_theta=1e6,
           eps=1e-6)


def _model():
    from cmf_amd import synth
    from cmf_amd.model import Model
    moe = dict(n_experts=64, top_k=8, inter=256, layers=[0, 1], router_dtype="q8")
    return Model(synth.synth_model(CFG, seed=31, norm_noise=0.1, sigma=0.05, mtp=False, moe=moe))


def test_scratch_follows_the_prompt(gpu):
    import ctypes as C

    from cmf_amd import synth
    hip = C.CDLL("libamdhip64.so.7")  # (the one the library is linked to)

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value
    m = _model()
    ids = synth.ids(32, 2100, CFG["vocab"])
    m.prefill(ids)  # (the thread's GEMM operands)
    m.free()
    m = _model()
    m.prefill(ids[:16])
    f0 = free()
    m.prefill(ids[:40])
    f1 = free()
    m.prefill(ids)
    f2 = free()
    m.free()
    print(f"16 -> 40 positions {(f0 - f1) >> 20} MiB, -> 2100 {(f1 - f2) >> 20} MiB", flush=True)
    # rows of a 64-row tile per expert and pair: 2 KiB of operand and 2 of
    # output each, 256 * 8 / 64 + 64 tiles and 2048 * 8 / 64 + 64
    small, full = (32 + 64) * 64 * 4096, (256 + 64) * 64 * 4096
    assert f0 - f1 <= small + (8 << 20)
    assert f1 - f2 >= full - small - (8 << 20)


CHILD = """
import sys
sys.path.insert(0, sys.argv[1])
sys.path.insert(0, sys.argv[1] + "/tests")
import numpy as np
import cmf_amd
from cmf_amd import synth
from conftest import rel_l2
from test_gpu_moe_prefill_scratch import CFG, _model
cmf_amd.init(0)
m = _model()
ids = synth.ids(33, 70, CFG["vocab"])
m.prefill(ids)
tip, kv = m.state()[1], m.kv_export(1, 70)
for p in range(0, 70, 16):
    hid, _ = m.forward_batch(ids[p:p + 16], p, want_logits=False)
print(max([rel_l2(tip, hid[-1])] + [rel_l2(a, b) for a, b in zip(kv, m.kv_export(1, 70))]))
"""


def test_refused_scratch_takes_batches(gpu):
    env = dict(os.environ, CMF_PREFILL_MOE_FAIL="1")
    r = subprocess.run([sys.executable, "-c", CHILD, ROOT], capture_output=True, text=True, timeout=100, env=env)
    assert r.returncode == 0, r.stderr[-2000:]
    assert float(r.stdout.split()[-1]) < 2e-5  # (as test_gpu_moe_prefill)

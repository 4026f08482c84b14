"""The prefill attention's two workgroups per long query block meet through
global memory: the one that publishes its sums (an exchange of the launch's
tag by one thread, after a workgroup barrier) must have had every wave's
stores finished before that barrier.  On gfx950 the barrier itself waits for
LDS only, so the wait has to stand in the code of all waves before it, and the
write-back of the L2 has to have ended before the exchange."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_partial_sums_are_out_before_they_are_published(tmp_path):
    out = tmp_path / "prefill_attn.s"
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "--offload-device-only", "-S", "-x", "hip",
                        os.path.join(ROOT, "cmf_amd", "csrc", "prefill_attn.hip"), "-o", str(out)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    kernels = re.findall(r"^(_Z\S*k_prefill_faI\S*):(.*?)\.Lfunc_end", out.read_text(), re.S | re.M)
    assert len(kernels) == 10
    for name, body in kernels:
        code = [l.strip() for l in body.splitlines()]
        published = 0
        for i, l in enumerate(code):
            if not l.startswith("global_atomic_swap_x2"):
                continue
            bar = max((j for j in range(i) if code[j].startswith("s_barrier")), default=None)
            if bar is None:  # (the placement check's exchange, at the kernel's start)
                continue
            store = max(j for j in range(bar) if code[j].startswith("global_store"))
            wait = [c for c in code[store + 1:bar] if c.startswith("s_waitcnt") and "vmcnt(0)" in c]
            assert wait, f"{name}: no wait for the stores before the barrier"
            back = max(j for j in range(i) if code[j].startswith("buffer_wbl2"))
            assert back > bar and any(c.startswith("s_waitcnt") and "vmcnt(0)" in c for c in code[back + 1:i]), name
            published += 1
        assert published == 1, name

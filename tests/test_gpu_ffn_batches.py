"""The FFN of more than 16 host rows in batches of 16 (what is left to rows
whose large-batch scratch does not fit) equals the large-batch GEMMs."""
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _ffn(dt):
    import cmf_amd
    from cmf_amd import synth
    mk = {"q8": synth.q8_uniform, "q4t": synth.q4t_uniform, "q4tp": synth.q4tp_uniform}[dt]
    ws = []
    for r, c, s in ((800, 288, 21), (800, 288, 22), (288, 800, 23)):
        t = mk(s, r, c)
        ws.append(cmf_amd.Weight(t["dtype"], r, c, payload=t["bytes"], q=t["q"], row_scale=t["row_scale"]))
    x = synth.normal(24, 53 * 288).reshape(53, 288) * np.float32(0.1)
    out = np.full((53, 288), np.nan, np.float32)
    assert cmf_amd.ffn(*ws, x, 53, 288, 800, out)
    return out


@pytest.mark.parametrize("dt", ["q8", "q4t", "q4tp"])
def test_batches_equal_gemms(gpu, dt, tmp_path):
    child = ("import sys; sys.path[:0] = [sys.argv[1], sys.argv[1] + '/tests']\nimport numpy as np\nimport cmf_amd\n"
             "from test_gpu_ffn_batches import _ffn\ncmf_amd.init(0)\nnp.save(sys.argv[3], _ffn(sys.argv[2]))\n")
    p = str(tmp_path / "out.npy")
    r = subprocess.run([sys.executable, "-c", child, ROOT, dt, p], capture_output=True, text=True, timeout=100,
                       env=dict(os.environ, CMF_FFN_GEMM="0"))
    assert r.returncode == 0, r.stderr[-2000:]
    # three products of 22-bit operands and f32 sums (5e-7 each) on each side
    assert rel_l2(_ffn(dt), np.load(p)) < 3e-6

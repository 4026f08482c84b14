"""A routed batch of a single (token, expert) pair: the job list holds one
job, whose expert is not the first one."""
import numpy as np
import pytest

from conftest import rel_l2
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("codec", ["q8", "q4t", "q4tp"])
def test_one_pair_uses_its_expert(gpu, codec):
    from cmf_amd import synth
    from cmf_amd.moe import MoE
    mk = {"q8": synth.q8_uniform, "q4t": synth.q4t_uniform, "q4tp": synth.q4tp_uniform}[codec]
    H, I, ne = 256, 128, 6
    ex = [{"gate": mk(50 + 3 * e, I, H), "up": mk(51 + 3 * e, I, H), "down": mk(52 + 3 * e, H, I)} for e in range(ne)]
    x = synth.normal(90, H).reshape(1, H)
    lg = np.zeros((1, ne), np.float32)
    lg[0, 4] = 3.0
    moe = MoE(ne, H, I, 1, ex)
    ref = orc.moe_ffn(ex, 1, lg[0], x[0], True, 1.0, threads=8)
    out, idx, _ = moe.ffn(x, lg)
    got = moe.block(x, [4], [1.0])
    print(f"{codec}: routed {rel_l2(out[0], ref):.1e}, caller-routed {rel_l2(got, ref):.1e}", flush=True)
    assert idx[0, 0] == 4
    assert rel_l2(out[0], ref) < 1e-3 and rel_l2(got, ref) < 1e-3
    moe.free()

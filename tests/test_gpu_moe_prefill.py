"""Prefill of routed-expert models: chunks of more than 16 rows run the
experts as grouped large-batch GEMMs over the pairs sorted by expert; the
same tokens in batches of 16 rows (forward_batch) take the verify-batch
kernels.  Both must leave the same keys, values and tip hidden row, for every
expert codec and router kind, chunks that leave part of a 64-row tile,
experts that no token picked and experts with several tiles."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

CFG = dict(n_layers=3, hidden=256, n_heads=4, n_kv=2, head_dim=128, inter=512, vocab=2048, max_seq=1400,
           rope_theta=1e6, eps=1e-6)


def _model(ffn, router, ne, k, inter):
    from cmf_amd import DT_Q4T, DT_Q8ROW, synth
    moe = dict(n_experts=ne, top_k=k, inter=inter, layers=[0, 2], router_dtype=router)
    sm = synth.synth_model(CFG, seed=31, norm_noise=0.1, sigma=0.05, mtp=False, moe=moe,
                           ffn_dtype=DT_Q8ROW if ffn == "q8" else DT_Q4T)
    if ffn == "q4tp":
        for li in (0, 2):
            for e, ex in enumerate(sm["layers"][li]["moe"]["experts"]):
                for i, (n, r, c) in enumerate((("gate", inter, 256), ("up", inter, 256), ("down", 256, inter))):
                    ex[n] = synth.q4tp_uniform(1000 * li + 10 * e + i, r, c, sigma=0.001)
    return sm


@pytest.mark.parametrize("ffn,router,ne,k,inter,n", [
    ("q4t", "f16", 16, 4, 128, 70), ("q4t", "q8", 5, 2, 96, 17), ("q4tp", "f16", 40, 3, 160, 130),
    ("q8", "q8", 16, 8, 128, 300), ("q8", "f16", 130, 1, 32, 33), ("q4tp", "q8", 2, 2, 64, 1100)])
def test_moe_prefill_equals_batches(gpu, ffn, router, ne, k, inter, n):
    from cmf_amd import synth
    from cmf_amd.model import Model
    m = Model(_model(ffn, router, ne, k, inter))
    ids = synth.ids(32, n, CFG["vocab"])
    m.prefill(ids)
    tip = m.state()[1]
    kv = [m.kv_export(li, n) for li in range(3)]
    for p in range(0, n, 16):
        hid, _ = m.forward_batch(ids[p:p + 16], p, want_logits=False)
    # one rounding of 22-bit operands and f32 sums a product (5e-7), ten of
    # them on the way to the last layer's keys, each passed on by the norms
    errs = [rel_l2(tip, hid[-1])] + [rel_l2(a, b) for li in range(3) for a, b in zip(kv[li], m.kv_export(li, n))]
    print(f"{ffn} {router} {ne}x{k} inter {inter} n={n}: tip {errs[0]:.1e}, keys and values {max(errs[1:]):.1e}", flush=True)
    assert max(errs) < 2e-5
    m.free()

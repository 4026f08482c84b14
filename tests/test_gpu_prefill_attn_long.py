"""The prefill attention on both sides of the context length at which its
query blocks grow from 64 to 128 rows (576 keys), at the edges of the
128-row blocks (a row more than a block, odd and even numbers of blocks, the
longer block of a pair in two halves, one and two query heads a KV head, one
KV head per XCD and placed by the grid).  The second layer's K / V rows see
the first layer's attention at every position; against the same tokens in
batches of 16 rows through the decode kernels."""
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv,n", [
    (8, 8, 576), (8, 8, 577), (4, 4, 641), (1, 1, 769), (8, 8, 1023),   # 128 positions a block
    (4, 2, 576), (16, 8, 577), (4, 2, 641), (16, 8, 705), (2, 1, 1024), (2, 1, 1025),  # 64
])
def test_prefill_attention_block_rows(gpu, heads, kv, n):
    from cmf_amd import synth
    from cmf_amd.model import Model
    cfg = dict(n_layers=2, hidden=256, n_heads=heads, n_kv=kv, head_dim=128, inter=256, vocab=512,
               max_seq=1152, rope_theta=1e6, eps=1e-6)
    m = Model(synth.synth_model(cfg, seed=31, norm_noise=0.1, sigma=0.05, mtp=False))
    ids = synth.ids(32, n, cfg["vocab"])
    m.prefill(ids)
    tip, kv1 = m.state()[1], m.kv_export(1, n)
    for p in range(0, n, 16):
        hid, _ = m.forward_batch(ids[p:p + 16], p, want_logits=False)
    worst = [rel_l2(tip, hid[-1])]
    for a, b in zip(kv1, m.kv_export(1, n)):
        worst += [rel_l2(a[:, c:c + 64], b[:, c:c + 64]) for c in range(0, n, 64)]
    print(f"{heads}/{kv} n={n}: {max(worst):.1e}", flush=True)
    # (both sides round 22-bit operands and sum in f32, in different orders; a
    # dropped or doubled key is above 1e-3)
    assert max(worst) < 1e-5
    m.free()

"""The prefill attention's query blocks of contexts up to 576 keys (64 rows of
a kv head's query heads, paired) at their edges: one and two query heads a kv
head, one row, a row more than a block or a pair of them, odd and even numbers
of blocks, one KV head per XCD (8 KV heads) and placed by the grid.  The second layer's K / V
rows see the first layer's attention at every position, so they are compared
with the oracle's per-position forwards in 64-row pieces, within the relative
L2 of 1e-4 that the prefill is held to everywhere (both sides sum in f32, in
different orders)."""
import pytest

from conftest import rel_l2
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv,n", [
    (1, 1, 1), (2, 2, 33), (8, 8, 129), (8, 8, 385),     # 64 positions a block
    (4, 2, 64), (4, 2, 65), (16, 8, 193),                # 32
    (16, 8, 321), (2, 1, 448),
])
def test_prefill_attention_block_edges(gpu, heads, kv, n):
    from cmf_amd import synth
    from cmf_amd.model import Model
    cfg = dict(n_layers=2, hidden=256, n_heads=heads, n_kv=kv, head_dim=128, inter=256, vocab=512,
               max_seq=512, rope_theta=1e6, eps=1e-6)
    sm = synth.synth_model(cfg, seed=31, norm_noise=0.1, sigma=0.05)
    g = Model(sm)
    o = orc.OracleModel(sm, threads=8)
    ids = synth.ids(32, n, cfg["vocab"])
    g.prefill(ids)
    otip = o.prefill(ids)
    _, tip = g.state()
    assert rel_l2(tip, otip) < 1e-4
    (k, v), (rk, rv) = g.kv_export(1, n), o.kv(1)
    for c0 in range(0, n, 64):
        for a, b in ((k, rk), (v, rv)):
            assert rel_l2(a[:, c0:c0 + 64], b[:, c0:c0 + 64]) < 1e-4, c0
    g.free()

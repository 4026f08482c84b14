"""The per-job expert GEMVs of every codec at batches up to 16: jobs of one
token and of more than one pass of token slots (q8 passes hold 5, q4 8), rows
of every instance's step count, ragged row blocks, mixed gate|up and down
codecs.  Against an f64 product of the dequantized experts with the device's
own routing."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _tensor(dt, seed, rows, cols):
    from cmf_amd import synth
    return {"q8": synth.q8_uniform, "q4t": synth.q4t_uniform, "q4tp": synth.q4tp_uniform}[dt](seed, rows, cols)


@pytest.mark.parametrize("gu,down,ne,k,H,I,b", [
    ("q8", "q8", 64, 8, 1024, 512, 16), ("q8", "q8", 2, 2, 256, 96, 16), ("q8", "q8", 7, 3, 544, 800, 11),
    ("q8", "q8", 12, 4, 2048, 768, 6), ("q4tp", "q4tp", 9, 4, 1056, 672, 16), ("q4tp", "q4tp", 32, 2, 2048, 1536, 5),
    ("q4t", "q4t", 3, 2, 512, 1056, 9), ("q4t", "q4t", 16, 8, 2048, 768, 16), ("q8", "q4t", 6, 2, 4096, 32, 13),
    ("q4tp", "q8", 5, 1, 320, 2080, 16), ("q4t", "q8", 4, 4, 4128, 64, 12)])
def test_moe_rows(gpu, gu, down, ne, k, H, I, b):
    from cmf_amd import synth
    from cmf_amd.moe import MoE
    ex = [{"gate": _tensor(gu, 700 + 3 * e, I, H), "up": _tensor(gu, 701 + 3 * e, I, H),
           "down": _tensor(down, 702 + 3 * e, H, I)} for e in range(ne)]
    x = synth.normal(71, b * H).reshape(b, H) * np.float32(0.05)
    moe = MoE(ne, H, I, k, ex)
    out, idx, w = moe.ffn(x, synth.normal(72, b * ne).reshape(b, ne))
    moe.free()
    ref, bound = np.zeros((b, H)), np.zeros((b, H))
    eps = lambda c: 2.0 ** -23 * (c // 32 + 16)  # noqa: E731
    for e in sorted(set(idx.ravel().tolist())):
        g, u, d = (synth.dequant(ex[e][n]).astype(np.float64) for n in ("gate", "up", "down"))
        t, rank = np.nonzero(idx == e)
        xt = x[t].astype(np.float64)
        a, c = xt @ g.T, xt @ u.T
        h = a / (1 + np.exp(-a)) * c
        wt = w[t, rank].astype(np.float64)[:, None]
        np.add.at(ref, t, wt * (h @ d.T))
        # 22-bit operands and f32 sums of each product, the first two through
        # a SiLU of slope at most 1.1
        eg, eu = (2.0 ** -22 * np.abs(xt).max(1)[:, None] * np.abs(m).sum(1) + eps(H) * (np.abs(xt) @ np.abs(m).T) for m in (g, u))
        eh = 1.1 * eg * np.abs(c) + np.abs(a) * eu + 2.0 ** -20 * np.abs(h)
        eb = eh @ np.abs(d).T + 2.0 ** -22 * np.abs(h).max(1)[:, None] * np.abs(d).sum(1) + eps(I) * (np.abs(h) @ np.abs(d).T)
        np.add.at(bound, t, wt * (eb + 2.0 ** -22 * np.abs(h @ d.T)))
    err = np.abs(out - ref)
    print(f"{gu}/{down} {ne}x{k} {H}/{I} b={b}: largest error / bound {np.max(err / bound):.3f}", flush=True)
    assert np.all(err <= bound)

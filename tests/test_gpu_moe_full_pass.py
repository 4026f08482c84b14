"""Expert GEMVs whose jobs fill a pass of token slots, at operand sizes that
are no whole number of 1 KiB copy chunks (an odd number of slots of an odd
number of 128-column steps, q8 rows of 12 nk items): the copy's last chunk
ends past the operand.  All tokens pick the same experts.  Against an f64
product of the dequantized experts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# (passes of 1, 3, 5, 7 slots; q4t of at most 8 tokens: k_moe_q4t)
@pytest.mark.parametrize("dt,ne,k,H,I,b", [
    ("q4tp", 2, 1, 1152, 96, 1), ("q4tp", 2, 1, 1152, 160, 3), ("q4tp", 2, 1, 640, 128, 5), ("q4tp", 2, 1, 1408, 96, 7),
    ("q4tp", 64, 8, 1152, 64, 12), ("q4t", 64, 8, 1152, 64, 12), ("q4t", 2, 1, 1152, 96, 1), ("q4t", 2, 1, 1920, 96, 3),
    ("q4t", 3, 2, 384, 128, 7), ("q8", 2, 1, 256, 64, 1), ("q8", 2, 1, 896, 96, 2), ("q8", 2, 2, 448, 64, 16)])
def test_jobs_of_a_full_pass(gpu, dt, ne, k, H, I, b):
    from cmf_amd import synth
    from cmf_amd.moe import MoE
    mk = {"q8": synth.q8_uniform, "q4t": synth.q4t_uniform, "q4tp": synth.q4tp_uniform}[dt]
    ex = [{"gate": mk(500 + 3 * e, I, H), "up": mk(501 + 3 * e, I, H), "down": mk(502 + 3 * e, H, I)} for e in range(ne)]
    x = synth.normal(61, b * H).reshape(b, H) * np.float32(0.05)
    lg = np.zeros((b, ne), np.float32)
    picks = np.arange(ne - k, ne)
    lg[:, picks] = 4 + np.arange(k, dtype=np.float32)[None, :] / 8
    moe = MoE(ne, H, I, k, ex)
    out, idx, w = moe.ffn(x, lg)
    again = moe.ffn(x, lg)[0]
    moe.free()
    assert np.array_equal(np.sort(idx, 1), np.tile(picks, (b, 1)))
    assert np.array_equal(out, again)
    xd = x.astype(np.float64)
    ref, bound = np.zeros((b, H)), np.zeros((b, H))
    eps = lambda c: 2.0 ** -23 * (c // 32 + 16)  # noqa: E731
    for e in picks:
        g, u, d = (synth.dequant(ex[e][n]).astype(np.float64) for n in ("gate", "up", "down"))
        a, c = xd @ g.T, xd @ u.T
        h = a / (1 + np.exp(-a)) * c
        wt = w[idx == e].astype(np.float64)[:, None]
        ref += wt * (h @ d.T)
        # 22-bit operands and f32 sums of each product, the first two through
        # a SiLU of slope at most 1.1
        eg, eu = (2.0 ** -22 * np.abs(xd).max(1)[:, None] * np.abs(m).sum(1) + eps(H) * (np.abs(xd) @ np.abs(m).T) for m in (g, u))
        eh = 1.1 * eg * np.abs(c) + np.abs(a) * eu + 2.0 ** -20 * np.abs(h)
        bound += wt * (eh @ np.abs(d).T + 2.0 ** -22 * np.abs(h).max(1)[:, None] * np.abs(d).sum(1)
                       + eps(I) * (np.abs(h) @ np.abs(d).T) + 2.0 ** -22 * np.abs(h @ d.T))
    err = np.abs(out - ref)
    print(f"{dt} {ne}x{k} {H}/{I} b={b}: largest error / bound {np.max(err / bound):.3f}", flush=True)
    assert np.all(err <= bound)

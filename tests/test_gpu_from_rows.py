"""GEMVs and FFNs from plain f32 rows: one-row GEMVs that stage their own
operand (q8, q4t) equal the operand producer plus the prepared-operand GEMV
bit for bit at every instance's step count, rows that no wide load fits keep
the general producer, and the FFN of more than 16 rows (large-batch GEMMs)
equals an f64 product."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _weight(gpu, dt, rows, cols, seed=3):
    from cmf_amd import synth
    t = {"q8": synth.q8_uniform, "q4t": synth.q4t_uniform, "q4tp": synth.q4tp_uniform}[dt](seed, rows, cols)
    return t, gpu.Weight(t["dtype"], rows, cols, payload=t["bytes"], q=t["q"], row_scale=t["row_scale"])


# q8: the last column count of each instance (8, 16, 32, 64, 128, 192 steps of
# 64), one step past it, a partial step, columns that are no multiple of 4
Q8_COLS = [4, 100, 512, 516, 1024, 1028, 2048, 2052, 4096, 4100, 8192, 8196, 12288, 12292, 1002]
Q4_COLS = [32, 512, 544, 1024, 2048, 4096, 4128, 8192, 8224]


@pytest.mark.parametrize("dt,cols", [("q8", c) for c in Q8_COLS] + [(d, c) for d in ("q4t", "q4tp") for c in Q4_COLS])
def test_one_row_equals_prepared(gpu, dt, cols):
    from cmf_amd import synth
    rows, L = 37, gpu.lib()
    t, w = _weight(gpu, dt, rows, cols)
    pl, xs = gpu.DevBuf(L.cmf_prep_bytes(w.h)), gpu.DevBuf(256)
    dx, dy = gpu.DevBuf((cols + 1) * 4), gpu.DevBuf(rows * 4)
    wd = synth.dequant(t).astype(np.float64)
    for x in (synth.normal(5, cols), np.zeros(cols, np.float32)):
        for off in (0, 1):  # (an odd address: no wide loads)
            buf = np.zeros(cols + 1, np.float32)
            buf[off:off + cols] = x
            dx.upload(buf)
            gpu.check(L.cmf_prep_dev(w.h, dx.p + 4 * off, cols, 1, pl.p, xs.p))
            gpu.check(L.cmf_gemv_prepared(w.h, pl.p, xs.p, 1, dy.p, rows, 0))
            gpu.check(L.cmf_sync())
            want = dy.download((rows,))
            gpu.check(L.cmf_gemv_dev_noalloc(w.h, dx.p + 4 * off, cols, 1, dy.p, rows))
            gpu.check(L.cmf_sync())
            assert np.array_equal(dy.download((rows,)), want)
            bound = 2.0 ** -22 * np.abs(x).max() * np.abs(wd).sum(1) + 2.0 ** -23 * (cols // 32 + 16) * (np.abs(wd) @ np.abs(x))
            assert np.all(np.abs(want - wd @ x.astype(np.float64)) <= bound)
    w.free()


# batches of a split producer (items past a workgroup's 256, a partial one)
@pytest.mark.parametrize("dt,cols,m", [("q4t", 2080, 13), ("q4tp", 4128, 9), ("q8", 4112, 16), ("q8", 1000, 6), ("q4t", 96, 2)])
def test_batch_rows(gpu, dt, cols, m):
    from cmf_amd import synth
    rows = 53
    t, w = _weight(gpu, dt, rows, cols, seed=9)
    x = synth.normal(6, m * cols).reshape(m, cols)
    got = gpu.matmul(w, x).astype(np.float64)
    wd, xd = synth.dequant(t).astype(np.float64), x.astype(np.float64)
    bound = (2.0 ** -22 * np.abs(xd).max(1)[:, None] * np.abs(wd).sum(1)[None, :]
             + 2.0 ** -23 * (cols // 32 + 16) * (np.abs(xd) @ np.abs(wd).T))
    assert np.all(np.abs(got - xd @ wd.T) <= bound)
    w.free()


@pytest.mark.parametrize("dt,hidden,inter,b", [("q4t", 256, 512, 17), ("q4tp", 288, 800, 65), ("q8", 320, 12320, 40),
                                               ("q8", 90, 130, 33), ("q4t", 64, 96, 2100)])
def test_ffn_large_batch(gpu, dt, hidden, inter, b):
    from cmf_amd import synth
    (t1, w1), (t3, w3), (t2, w2) = (_weight(gpu, dt, r, c, s) for r, c, s in
                                    ((inter, hidden, 21), (inter, hidden, 22), (hidden, inter, 23)))
    x = synth.normal(24, b * hidden).reshape(b, hidden) * np.float32(0.1)
    out = np.empty((b, hidden), np.float32)
    assert gpu.ffn(w1, w3, w2, x, b, hidden, inter, out)
    d1, d3, d2 = (synth.dequant(t).astype(np.float64) for t in (t1, t3, t2))
    g, u = x @ d1.T, x @ d3.T
    h = g / (1 + np.exp(-g)) * u
    ref = h @ d2.T
    # three products of 22-bit operands and f32 sums, the first two through a
    # SiLU of slope at most 1.1
    eg, eu = (2.0 ** -22 * np.abs(x).max(1)[:, None] * np.abs(d).sum(1) + 2.0 ** -23 * (hidden // 32 + 16) * (np.abs(x) @ np.abs(d).T)
              for d in (d1, d3))
    eh = 1.1 * eg * np.abs(u) + np.abs(g) * eu + 2.0 ** -20 * np.abs(h)
    bound = (eh @ np.abs(d2).T + 2.0 ** -22 * np.abs(h).max(1)[:, None] * np.abs(d2).sum(1)
             + 2.0 ** -23 * (inter // 32 + 16) * (np.abs(h) @ np.abs(d2).T))
    err = np.abs(out - ref)
    print(f"{dt} {hidden}/{inter} b={b}: largest error / bound {np.max(err / bound):.3f}", flush=True)
    assert np.all(err <= bound)
    for w in (w1, w3, w2):
        w.free()


@pytest.mark.parametrize("attn,ffn,H,I,n", [("q8", "q4t", 256, 512, 9), ("q8", "q8", 320, 608, 5), ("q4t", "q4t", 1056, 544, 5),
                                            ("q8", "q4t", 2048, 6144, 3)])
def test_one_row_blocks_equal_batches(gpu, attn, ffn, H, I, n):
    """one-row decoder blocks (the norm and the SwiGLU inside the one-row
    GEMVs) leave the rows that batches of rows (the general kernels) leave"""
    from cmf_amd import DT_Q4T, DT_Q8ROW, synth
    from cmf_amd.model import Model
    cfg = dict(n_layers=2, hidden=H, n_heads=2, n_kv=1, head_dim=128, inter=I, vocab=512, max_seq=64, rope_theta=1e6, eps=1e-6)
    dt = {"q8": DT_Q8ROW, "q4t": DT_Q4T}
    m = Model(synth.synth_model(cfg, seed=41, norm_noise=0.1, sigma=0.05, mtp=False, attn_dtype=dt[attn], ffn_dtype=dt[ffn]))
    ids = synth.ids(42, n, 512)
    rows = np.concatenate([m.forward_batch(ids[p:p + 1], p, want_logits=False)[0] for p in range(n)])
    both, lg = m.forward_batch(ids, 0)
    one = m.forward_batch(ids[n - 1:], n - 1)[1]
    err = np.linalg.norm(rows - both) / np.linalg.norm(both)
    print(f"{attn}/{ffn} {H}/{I}: rows {err:.1e}", flush=True)
    # seven products of 22-bit operands and f32 sums a layer (5e-7 each)
    assert err < 1e-5
    assert np.linalg.norm(one[0] - lg[-1]) < 1e-5 * np.linalg.norm(lg[-1])
    m.free()


@pytest.mark.parametrize("pos", [2040, 2047, 2049, 4300, 8191, 8300])
def test_long_context_merge(gpu, pos):
    """attention over more than 32 chunks of 64 positions (several waves merge
    them), against an f64 softmax over the exported keys and values"""
    from cmf_amd import synth
    from cmf_amd.model import Model
    cfg = dict(n_layers=1, hidden=256, n_heads=2, n_kv=1, head_dim=128, inter=64, vocab=512, max_seq=8400, rope_theta=1e6, eps=1e-6)
    sm = synth.synth_model(cfg, seed=43, norm_noise=0.1, sigma=0.05, mtp=False)
    for n in ("gate", "up", "down"):
        sm["layers"][0][n]["bytes"][:] = np.tile(np.array([0, 0] + [0x88] * 16, np.uint8), sm["layers"][0][n]["bytes"].size // 18)
    m = Model(sm)
    m.prefill(synth.ids(44, pos, 512))
    tok = synth.ids(45, 1, 512)
    hid, _ = m.forward_batch(tok, pos, want_logits=False)
    k, v = (a[0].astype(np.float64) for a in m.kv_export(0, pos + 1))
    m.free()
    l, lm = sm["layers"][0], sm["lm_head"]
    h = lm["q"][tok[0]].astype(np.float64) * lm["row_scale"][tok[0]]
    rms = lambda x, w: x / np.sqrt((x * x).mean(-1, keepdims=True) + 1e-6) * w  # noqa: E731
    q = rms((synth.dequant(l["wq"]).astype(np.float64) @ rms(h, l["input_norm"])).reshape(2, 128), l["q_norm"])
    ang = (np.float32(pos) * (np.float32(1) / np.power(np.float32(1e6), np.arange(64, dtype=np.float32) / np.float32(64)))).astype(np.float64)
    q = np.concatenate([q[:, :64] * np.cos(ang) - q[:, 64:] * np.sin(ang), q[:, :64] * np.sin(ang) + q[:, 64:] * np.cos(ang)], 1)
    s = q @ k.T / np.sqrt(128.0)
    p = np.exp(s - s.max(1, keepdims=True))
    o = (p / p.sum(1, keepdims=True)) @ v
    ref = h + synth.dequant(l["wo"]).astype(np.float64) @ o.reshape(-1)
    err = np.linalg.norm(hid[0] - ref) / np.linalg.norm(ref)
    print(f"position {pos}: {err:.1e}", flush=True)
    # the angles' frequencies are one ulp from the host's: pos * 2^-24 in the scores
    assert err < 1e-5 + pos * 2.0 ** -24


@pytest.mark.parametrize("cols", [2560, 2592, 2720, 2752])
def test_operand_at_the_lds_limit(gpu, cols):
    """16 q8 rows whose planes just fit, do not fit beside the kernel's static
    LDS, and are past the budget"""
    from cmf_amd import synth
    t, w = _weight(gpu, "q8", 40, cols)
    x = synth.normal(8, 16 * cols).reshape(16, cols)
    got, ref = gpu.matmul(w, x).astype(np.float64), x.astype(np.float64) @ synth.dequant(t).astype(np.float64).T
    assert np.linalg.norm(got - ref) < 2e-6 * np.linalg.norm(ref)
    w.free()

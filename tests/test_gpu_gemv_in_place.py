"""A GEMV whose result overlaps its operand row: y over x, or shifted against
it by a few rows, gives what a result buffer of its own gives."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b", [1, 3])
@pytest.mark.parametrize("dt", ["q8", "q4t", "q4tp"])
def test_result_over_operand(gpu, dt, b):
    from cmf_amd import synth
    n, L = 4096, gpu.lib()
    t = {"q8": synth.q8_uniform, "q4t": synth.q4t_uniform, "q4tp": synth.q4tp_uniform}[dt](3, n, n)
    w = gpu.Weight(t["dtype"], n, n, payload=t["bytes"], q=t["q"], row_scale=t["row_scale"])
    x = synth.normal(5, b * n)
    dx, dy = gpu.DevBuf((b * n + 128) * 4), gpu.DevBuf(b * n * 4)
    for xo, yo in ((0, 0), (0, 64), (64, 0)):
        buf = np.zeros(b * n + 128, np.float32)
        buf[xo:xo + b * n] = x
        dx.upload(buf)
        gpu.check(L.cmf_gemv_dev_noalloc(w.h, dx.p + 4 * xo, n, b, dy.p, n))
        gpu.check(L.cmf_gemv_dev_noalloc(w.h, dx.p + 4 * xo, n, b, dx.p + 4 * yo, n))
        gpu.check(L.cmf_sync())
        assert np.array_equal(dx.download((b * n + 128,))[yo:yo + b * n], dy.download((b * n,)))
    w.free()

"""The large-batch GEMM (batches above 16 rows) and its operand producers at
the edges of their tiles: row counts that leave part of a 16-row block, a
wave's 32 / 64 rows or a workgroup, column counts that leave part of a group
of tiles or of a 64-column chunk, one K part and several, 32 weight rows a
wave (test_gpu_gemm_rules has 64), and rows that the wave-per-row producer
holds or that take the general one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# rows, cols, batch: (q4) one part / split K; the last
# two: the most columns the wave-per-row producer holds, and past it
Q4 = [(1000, 1056, 77), (16, 32, 17), (48, 160, 64), (2064, 512, 1030), (3072, 128, 700), (24, 8192, 33), (8, 8224, 18)]
Q8 = [(1000, 1056, 77), (16, 48, 17), (40, 100, 65), (272, 1000, 130), (4112, 192, 1100), (24, 8192, 33), (8, 8208, 18)]


def _tensor(dt, rows, cols):
    from cmf_amd import synth
    if dt == "q8":
        return synth.q8_uniform(11, rows, cols)
    return (synth.q4t_uniform if dt == "q4t" else synth.q4tp_uniform)(12, rows, cols)


@pytest.mark.parametrize("dt,shape", [(d, s) for d in ("q4t", "q4tp") for s in Q4] + [("q8", s) for s in Q8])
def test_gemm_edges(gpu, dt, shape):
    from cmf_amd import synth
    rows, cols, m = shape
    t = _tensor(dt, rows, cols)
    x = synth.normal(13, m * cols).reshape(m, cols) * np.exp2(np.arange(m) % 7 - 3, dtype=np.float32)[:, None]
    x[m // 2] = 0.0  # a row without a largest value
    w = gpu.Weight(t["dtype"], rows, cols, payload=t["bytes"], q=t["q"], row_scale=t["row_scale"])
    got = gpu.matmul(w, x).astype(np.float64)
    w.free()
    wd, xd = synth.dequant(t).astype(np.float64), x.astype(np.float64)
    ref = xd @ wd.T
    # the operand's rounding (22 bits of the row's largest value), and one f32
    # rounding per tile (q4) or per plane and part (q8) of what is summed
    sums = cols // 32 + 8 if dt != "q8" else 16
    bound = (2.0 ** -22 * np.abs(xd).max(1)[:, None] * np.abs(wd).sum(1)[None, :]
             + 2.0 ** -23 * sums * (np.abs(xd) @ np.abs(wd).T))
    err = np.abs(got - ref)
    print(f"{dt} {rows}x{cols} m={m}: largest error / bound {np.max(err / np.maximum(bound, 1e-30)):.3f}", flush=True)
    assert np.all(err <= bound)
    assert np.all(got[m // 2] == 0.0)

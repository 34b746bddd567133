"""Two fields that share a complex x transform share its round-off only up to
2^10 of their ratio.  With the buoyancy off the scalar is passive, so a scalar
scaled by a power of two (exact in everything it enters) has to leave the
velocities of a large-eddy simulation as they were, and to come out scaled:
within 4 * 2^10 eps of the largest value, and bit for bit between two scales
that are both far off.  Rows of threads that divide a wavefront and rows that do
not."""
import numpy as np
import pytest

from diablo_amd import case, gpu

pytestmark = pytest.mark.gpu

FLOW = ("CU1", "CU2", "CU3")


def run(size, s):
    cfg = case.channel_case(*size, kick=0.3, streak=0.1)
    cfg.ri = [0.0] * len(cfg.ri)
    u1, u2, u3, th = case.initial_physical(cfg)
    cfg.th_bc_ymin_c1 = [s * x for x in cfg.th_bc_ymin_c1]
    cfg.th_bc_ymax_c1 = [s * x for x in cfg.th_bc_ymax_c1]
    g = gpu.GpuChannel(cfg)
    g.initialize(u1, u2, u3, [s * t for t in th])
    g.set_les(True, True)
    g.step(2)
    out = g.state()
    g.close()
    return out


@pytest.mark.parametrize("size", [(96, 11, 16), (54, 9, 18), (128, 9, 16), (384, 8, 8)])
def test_scales_of_a_pair(size):
    print(size, flush=True)
    tol = 4 * 2 ** 10 * np.finfo(float).eps
    one = run(size, 1.0)
    assert np.abs(one["CTH0"]).max() > 0
    for e in (30, -30):
        s = 2.0 ** e
        far = run(size, s)
        for k, t in [(k, 1.0) for k in FLOW] + [("CTH0", s)]:
            err = np.abs(far[k] - t * one[k]).max() / np.abs(t * one[k]).max()
            print(e, k, err, flush=True)
            assert err <= tol, (e, k, err)
    a, b = run(size, 2.0 ** 30), run(size, 2.0 ** 40)
    for k in FLOW + ("CP", "CF1", "CF2", "CF3"):
        assert np.array_equal(a[k], b[k]), k

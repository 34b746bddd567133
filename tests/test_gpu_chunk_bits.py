"""How many planes a block of the x kernel takes, and whether it runs for one
context or for an ensemble's batch, does not change a bit of the results: every
length that has a compile-time plan, and two that have none."""
import numpy as np
import pytest

from diablo_amd import case, gpu

pytestmark = pytest.mark.gpu

SIZES = [(64, 17, 24), (96, 17, 24), (128, 17, 24), (192, 17, 24), (256, 17, 24), (384, 17, 24), (54, 17, 24),
         (162, 17, 24)]
FIELDS = ("CU1", "CU2", "CU3", "CP", "CTH0", "CF1", "CF2", "CF3", "CFTH0")


def _same(a, b, what):
    for k in FIELDS:
        assert np.array_equal(a[k], b[k]), (what, k, np.abs(a[k] - b[k]).max() / np.abs(b[k]).max())


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("size", SIZES)
def test_bits_of_the_x_kernel(monkeypatch, size, precision):
    nx, ny, nz = size
    print(size, precision, flush=True)
    monkeypatch.delenv("DGPU_XCHUNK", raising=False)
    cfgs = [case.channel_case(nx, n, nz, kick=0.3, streak=0.1) for n in (ny, ny + 4)]
    start = [case.initial_physical(c) for c in cfgs]

    def run(chunk):
        if chunk:
            monkeypatch.setenv("DGPU_XCHUNK", str(chunk))
        g = gpu.GpuChannel(cfgs[0], precision=precision)
        g.initialize(*start[0])
        g.step(2)
        s = g.state()
        g.close()
        return s

    ref = run(0)
    for chunk in (1, 2, 3, 5, 8, 64):
        _same(run(chunk), ref, chunk)
    monkeypatch.delenv("DGPU_XCHUNK", raising=False)
    ens = gpu.GpuEnsemble(cfgs, precision=precision)
    for m, p in zip(ens.members, start):
        m.initialize(*p)
    ens.step(2)
    ens.synchronize()
    _same(ens.members[0].state(), ref, "ensemble")
    ens.close()


@pytest.mark.parametrize("size", SIZES)
def test_f64state_keeps_its_accuracy(monkeypatch, size):
    """mixed_f64state runs have x kernels of their own, whose bits may depend on
    the planes per block: the state stays within FP32 round-off of the nonlinear
    terms (64 eps of them, and they move the state by at most a tenth of itself
    in two steps: 8e-7) of the FP64 run for any number of planes."""
    nx, ny, nz = size
    print(size, flush=True)
    cfg = case.channel_case(nx, ny, nz, kick=0.3, streak=0.1)
    start = case.initial_physical(cfg)

    def run(precision, chunk):
        if chunk:
            monkeypatch.setenv("DGPU_XCHUNK", str(chunk))
        else:
            monkeypatch.delenv("DGPU_XCHUNK", raising=False)
        g = gpu.GpuChannel(cfg, precision=precision)
        g.initialize(*start)
        g.step(2)
        s = g.state()
        g.close()
        return s

    ref = run("fp64", 0)
    for chunk in (0, 1, 3, 64):
        s = run("mixed_f64state", chunk)
        for k in ("CU1", "CU3", "CTH0"):
            err = np.linalg.norm(s[k] - ref[k]) / np.linalg.norm(ref[k])
            assert err <= 8e-7, (chunk, k, err)

"""DGPU_FFT_EX asks for a number of values per thread of the x transforms.
Every number that a context accepts has to give the run's numbers: the default
plan's bits where the request falls back to it or is the default, and round-off
of two FP64 transforms of the row's largest value elsewhere."""
import numpy as np
import pytest

from diablo_amd import case, gpu

pytestmark = pytest.mark.gpu


def _results(cfg):
    g = gpu.GpuChannel(cfg)
    g.initialize(*case.initial_physical(cfg))
    g.poisson_p_chan()
    out = {"P": g.state()["CP"], "NU_T": g.les_chan()}
    g.step(1)
    out.update(g.state())
    g.close()
    return out


@pytest.mark.parametrize("ex,same", [(16, True), (8, True), (4, False)])
def test_values_per_thread(monkeypatch, ex, same):
    cfg = case.channel_case(64, 17, 32, kick=0.3, streak=0.1)
    print("EX", ex, flush=True)
    monkeypatch.delenv("DGPU_FFT_EX", raising=False)
    want = _results(cfg)
    monkeypatch.setenv("DGPU_FFT_EX", str(ex))
    got = _results(cfg)
    for k in want:
        if same:
            assert np.array_equal(got[k], want[k]), k
        else:
            assert np.abs(got[k] - want[k]).max() <= 1e-11 * np.abs(want[k]).max(), k

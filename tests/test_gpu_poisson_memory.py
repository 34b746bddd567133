"""POISSON_P_CHAN runs once a start: what it leaves allocated is bounded by 256
MB whatever the run's size, and its result does not depend on where its planes
lie (NY around the edges of the runs of rows that a large run is cut into;
against the oracle with the bound of the same call's other tests)."""
import numpy as np
import pytest

from diablo_amd import case, gpu
from gpu_util import compare_states

pytestmark = pytest.mark.gpu


def _driver_mappings():
    """Bytes of this process that the GPU driver maps: device and pinned memory."""
    total = 0
    for line in open("/proc/self/maps"):
        f = line.split()
        if len(f) > 5 and "/dev/dri/" in f[5]:
            a, b = (int(x, 16) for x in f[0].split("-"))
            total += b - a
    return total


@pytest.mark.parametrize("size", [(192, 129, 192), (256, 257, 128)])
def test_memory_kept(size):
    print(size, flush=True)
    cfg = case.channel_case(*size, kick=0.3)
    g = gpu.GpuChannel(cfg)
    g.set_field(gpu.CU1, np.zeros(cfg.field_shape()))
    before = _driver_mappings()
    if not before:
        pytest.skip("no driver mappings to be read in /proc/self/maps")
    g.poisson_p_chan()
    grown = _driver_mappings() - before
    print("grown by", grown >> 20, "MiB", flush=True)
    assert grown <= (256 + 8) << 20
    g.close()


@pytest.mark.parametrize("size", [(192, 65, 256), (192, 66, 256), (192, 67, 256), (384, 22, 384), (384, 18, 384)])
def test_runs_of_rows(oracle_mod, size):
    print(size, flush=True)
    cfg = case.channel_case(*size, kick=0.3, streak=0.1)
    o = oracle_mod.Oracle(cfg)
    o.initialize(*case.initial_physical(cfg))
    g = gpu.GpuChannel(cfg)
    g.load_state(o.state())
    g.poisson_p_chan()
    o.poisson_p_chan()
    errs, bad = compare_states(cfg, g.state(), o.state(), 1e-11, fields=("CP",))
    print(errs, flush=True)
    assert not bad, bad
    g.close()

"""The pair-plane transforms and the kernels on them (LES, POISSON_P_CHAN) at
the sizes where they can go wrong: rows whose threads do not divide a
wavefront, every number of values per thread, rows wider than a block of 256
threads, a few planes, more planes than one chunk, and lengths only the mixed
contexts plan for.  Against the oracle; the bounds are those of the same
quantities elsewhere: FP64 round-off of transforms and of the strain's
differences, 1e-12 of the largest NU_T and 1e-11 of the largest force."""
import numpy as np
import pytest

from diablo_amd import case
from gpu_util import compare_states

pytestmark = pytest.mark.gpu

SIZES = [(16, 8, 12), (24, 9, 8), (54, 7, 18), (64, 40, 8), (96, 11, 16), (162, 6, 8), (256, 9, 8), (384, 8, 8),
         (512, 6, 8)]


def say(*a):
    print(*a, flush=True)


def _pair(oracle_mod, cfg, precision):
    from diablo_amd import gpu
    o = oracle_mod.Oracle(cfg)
    o.initialize(*case.initial_physical(cfg))
    o.step()
    g = gpu.GpuChannel(cfg, precision=precision)
    g.load_state(o.state())
    g.time = o.time
    return o, g


def _les_chan(oracle_mod, cfg, precision="fp64"):
    o, g = _pair(oracle_mod, cfg, precision)
    before = [case.kept(cfg, o.state()[k]).copy() for k in ("CF1", "CF2", "CF3")]
    a, b = g.les_chan(), o.les_chan()
    e = np.abs(a - b).max() / np.abs(b).max()
    say("NU_T", e)
    assert e < 1e-12
    sg, so = g.state(), o.state()
    for k, f in zip(("CF1", "CF2", "CF3"), before):
        ref = case.kept(cfg, so[k]) - f
        e = np.abs(case.kept(cfg, sg[k]) - f - ref).max() / np.abs(ref).max()
        say(k, e)
        assert e < 1e-11, k


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("deck", ["channel", "kh"])
def test_les_sizes(oracle_mod, size, deck):
    nx, ny, nz = size
    cfg = (case.channel_case(nx, ny, nz, kick=0.3, streak=0.1) if deck == "channel"
           else case.kh_case(nx, ny, nz, kick=0.05))
    say("les", deck, size)
    _les_chan(oracle_mod, cfg)
    o, g = _pair(oracle_mod, cfg, "fp64")
    o.set_les(True, True)
    g.set_les(True, True)
    o.step()
    g.step(1)
    g.synchronize()
    errs, bad = compare_states(cfg, g.state(), o.state(), 1e-11,
                               fields=("CU1", "CU2", "CU3", "CTH0", "CF1", "CF2", "CF3", "CFTH0"))
    say(errs)
    assert not bad, bad


@pytest.mark.parametrize("nx", [1024])
def test_les_chan_mixed_only_lengths(oracle_mod, nx):
    say("les_chan mixed", nx)
    _les_chan(oracle_mod, case.channel_case(nx, 6, 8, kick=0.3, streak=0.1), "mixed")


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("deck", ["channel", "kh"])
def test_poisson_sizes(oracle_mod, size, deck):
    """Odd and even NY (the last pair of rows half empty or full), more and
    fewer rows than the solve's 16 segments; 1e-11 as the same call's other test."""
    nx, ny, nz = size
    cfg = (case.channel_case(nx, ny, nz, kick=0.3, streak=0.1) if deck == "channel"
           else case.kh_case(nx, ny, nz, kick=0.05))
    say("poisson", deck, size)
    o, g = _pair(oracle_mod, cfg, "fp64")
    g.poisson_p_chan()
    o.poisson_p_chan()
    errs, bad = compare_states(cfg, g.state(), o.state(), 1e-11, fields=("CP",))
    say(errs)
    assert not bad, bad


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_many_mode_column_default(precision):
    """From 8192 modes up the default column stage is the fused kernel at any
    NY it fits, below that not (NY = 150: the case that neither rule of short
    and tall columns covers).  FP64: within 1e-11 of the two kernels.  FP32
    state: no further from the FP64 run than 1.5 times the two kernels,
    plus 1e-7."""
    from diablo_amd import gpu

    def run(n, precision, shape=None):
        cfg = case.channel_case(n, 150, n, kick=0.05, dt=1e-4)
        say(n, precision, shape)
        g = gpu.GpuChannel(cfg, precision=precision)
        if shape is not None:
            g.set_column_shape(*shape)
        fused = g.column_fused()
        g.initialize(*case.initial_physical(cfg))
        g.step(1)
        g.synchronize()
        s = g.state()
        g.close()
        return cfg, fused, s

    assert not run(162, precision)[1]
    cfg, fused, one = run(192, precision)
    assert fused
    _, fused, two = run(192, precision, (8, 0))
    assert not fused
    if precision == "fp64":
        errs, bad = compare_states(cfg, one, two, 1e-11, ["CU1", "CU2", "CU3", "CP"])
        assert not bad, errs
        return
    ref = run(192, "fp64", (8, 0))[2]
    e1 = compare_states(cfg, one, ref, 1.0, ["CU1", "CU2", "CU3", "CP"])[0]
    e2 = compare_states(cfg, two, ref, 1.0, ["CU1", "CU2", "CU3", "CP"])[0]
    say("fused", e1, "two", e2)
    assert all(e1[k] <= 1.5 * e2[k] + 1e-7 for k in e1)

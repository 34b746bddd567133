"""The planes per block of an ensemble's batched x kernel: a few short members
get blocks for every CU, as a single run does, and a member keeps the shape of
its own for the calls it makes alone.  Bounds: 1.25 times the best of a few
shapes, where a fixed 64 planes (32 mixed) took 3.1 (2.1) times it."""
import time

import pytest

from diablo_amd import case, gpu

pytestmark = pytest.mark.gpu


def best_of(g, n=20):
    best = 1e9
    for _ in range(5):
        t = time.perf_counter()
        g.step(n)
        g.synchronize()
        best = min(best, (time.perf_counter() - t) / n)
    return best * 1e6


def _ensemble(precision):
    cfgs = [case.channel_case(64, ny, 64, kick=0.05, dt=1e-4) for ny in (33, 65, 97)]
    ens = gpu.GpuEnsemble(cfgs, precision=precision)
    for m, cfg in zip(ens.members, cfgs):
        m.initialize(*case.initial_physical(cfg))
    ens.step(3)
    ens.synchronize()
    return ens


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_small_group(monkeypatch, precision):
    us = {}
    for chunk in (0, 2, 4, 8):
        if chunk:
            monkeypatch.setenv("DGPU_XCHUNK", str(chunk))
        else:
            monkeypatch.delenv("DGPU_XCHUNK", raising=False)
        ens = _ensemble(precision)
        us[chunk] = best_of(ens)
        ens.close()
    print(precision, us, flush=True)
    assert us[0] <= 1.25 * min(us[c] for c in (2, 4, 8))


def test_member_alone(monkeypatch):
    monkeypatch.delenv("DGPU_XCHUNK", raising=False)
    ens = _ensemble("fp64")
    inside = best_of(ens.members[1])
    cfg = ens.members[1].cfg
    ens.close()
    g = gpu.GpuChannel(cfg)
    g.initialize(*case.initial_physical(cfg))
    g.step(3)
    alone = best_of(g)
    g.close()
    print(inside, alone, flush=True)
    assert inside <= 1.25 * alone

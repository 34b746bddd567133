"""Pinned memory of the host entry points: the members of an ensemble share one
set of slots (8 of 2 MiB), however many of them exchange fields, and the fields
come back as they were set, also when the calls come from several threads."""
import threading

import numpy as np
import pytest

from diablo_amd import case, gpu

pytestmark = pytest.mark.gpu

CFG = case.channel_case(192, 48, 192)


def _driver_mappings():
    """Bytes of this process that the GPU driver maps: device and pinned memory."""
    total = 0
    for line in open("/proc/self/maps"):
        f = line.split()
        if len(f) > 5 and "/dev/dri/" in f[5]:
            a, b = (int(x, 16) for x in f[0].split("-"))
            total += b - a
    return total


def _kept(a):
    return case.fourier_view(a)[:, :CFG.tnkz + 1, :CFG.nkx + 1]


def test_members_share_the_slots():
    warm = gpu.GpuChannel(CFG)
    a = np.zeros(CFG.field_shape())
    warm.set_field(gpu.CU1, a)
    ens = gpu.GpuEnsemble([CFG] * 8, precision="fp64")
    before = _driver_mappings()
    if not before:
        pytest.skip("no driver mappings to be read in /proc/self/maps")
    for m in ens.members:
        m.set_field(gpu.CU1, a)
    grown = _driver_mappings() - before
    print("grown by", grown >> 20, "MiB", flush=True)
    assert grown <= 2 * 8 * (2 << 20)
    ens.close()
    warm.close()


def test_members_from_several_threads():
    ens = gpu.GpuEnsemble([CFG] * 4, precision="fp64")
    rng = np.random.default_rng(5)
    fields = [rng.standard_normal(CFG.field_shape()) for _ in ens.members]
    got = [None] * len(fields)

    def work(i):
        for _ in range(4):
            ens.members[i].set_field(gpu.CU1, fields[i])
            got[i] = ens.members[i].get_field(gpu.CU1)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(fields))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i, f in enumerate(fields):
        assert np.array_equal(_kept(got[i]), _kept(f)), i
    ens.close()

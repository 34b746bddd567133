"""The host entry points that move the caller's arrays in chunks of planes:
one chunk, several chunks with a short last one, more chunks than workers and
planes larger than a chunk.  A field comes back as it was set, bit for bit,
with zeros in every slot that is not kept; a transform of all planes gives the
bits of plane-by-plane calls, and what lies outside the range stays."""
import numpy as np
import pytest

from diablo_amd import case, gpu

pytestmark = pytest.mark.gpu

# planes of 0.02, 0.3, 0.3, 0.6 and 2.1 MB
SIZES = [(64, 9, 32), (192, 17, 192), (192, 64, 192), (256, 33, 288), (512, 6, 512)]


def _chan(n):
    print(n, flush=True)
    cfg = case.channel_case(*n, kick=0.05)
    return cfg, gpu.GpuChannel(cfg), np.random.default_rng(7)


@pytest.mark.parametrize("n", SIZES)
def test_field_round_trip(n):
    cfg, g, rng = _chan(n)
    a = [rng.standard_normal(cfg.field_shape()) for _ in range(2)]
    for f, x in zip((gpu.CU1, gpu.CF2), a):
        g.set_field(f, x)
    for f, x in zip((gpu.CU1, gpu.CF2), a):
        b = np.full(cfg.field_shape(), np.nan)
        assert g.L.dgpu_get_field(g.h, f, gpu._dp(b)) == 0
        want = np.zeros_like(x)
        case.fourier_view(want)[:, :cfg.tnkz + 1, :cfg.nkx + 1] = \
            case.fourier_view(x)[:, :cfg.tnkz + 1, :cfg.nkx + 1]
        assert np.array_equal(b, want)
    g.close()


@pytest.mark.parametrize("n", SIZES)
def test_transforms_in_chunks(n):
    cfg, g, rng = _chan(n)
    a = rng.standard_normal(cfg.field_shape())
    lo, hi = 1, cfg.ny
    for fn in (g.fft_xz_to_fourier, g.fft_xz_to_physical):
        one, all_ = a.copy(), a.copy()
        fn(all_, lo, hi)
        for j in range(lo, hi + 1):
            fn(one, j, j)
        assert np.array_equal(one, all_)
        assert np.array_equal(all_[:lo], a[:lo]) and np.array_equal(all_[hi + 1:], a[hi + 1:])
    # the last call was to physical space: the rows beyond NZ are the caller's
    assert np.array_equal(all_[:, cfg.nz:], a[:, cfg.nz:])
    # and back and forth the kept modes come back (round-off of two transforms)
    f = a.copy()
    g.fft_xz_to_fourier(f, 0, cfg.ny + 1)
    p = f.copy()
    g.fft_xz_to_physical(p, 0, cfg.ny + 1)
    g.fft_xz_to_fourier(p, 0, cfg.ny + 1)
    assert np.abs(p - f).max() <= 1e-14 * np.sqrt(cfg.nx * cfg.nz) * np.abs(f).max()
    g.close()

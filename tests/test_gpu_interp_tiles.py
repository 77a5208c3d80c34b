"""Interpolation at the edges of its per-tile loops: tiles with point counts around the wave, the workgroup, the batches
of the ordering pass and its cap (2048 points, above which the binned order stays), tiles on both poles and the longitude
seam, a grid narrower than a tile, an even and an odd kernel polynomial degree, outer cells of higher degree than the
others, against direct summation.

Tolerance, relative 2-norm: ten times epsilon, as in the other comparisons of nusht2d2 with direct summation (thirty times
with the FP32 grid, epsilon >= 1e-6)."""
import numpy as np
import pytest
import torch

from oracle import almutil, sht as osht

pytestmark = pytest.mark.gpu

COUNTS = [1, 15, 16, 17, 63, 65, 255, 256, 257, 1023, 1024, 1025, 2047, 2048, 2049, 2500]


def _run(L, eps, sigma, loc, rng, spin):
    import cunusht_amd
    T = cunusht_amd.get_transformer("GPU")(("gl", {"lmax": L}), nuFFTtype=2, epsilon=eps, spin=spin, sigma=sigma)
    a = almutil.random_alm(L, spin, 1 if spin == 0 else 2, rng)
    at = torch.as_tensor(a[0] if spin == 0 else a, device="cuda")
    got = T.nusht2d2(L, L, at, torch.as_tensor(loc, device="cuda"), spin=spin).cpu().numpy()
    assert all(7 <= p.info()["kernel_width"] <= 16 for p in T._plans.values())  # the unrolled widths with paired cells
    ref = osht.synth_direct(a, L, spin, loc[:, 0], loc[:, 1])
    got = got if spin == 0 else got[0] + 1j * got[1]
    err = np.linalg.norm(got.reshape(-1) - ref) / np.linalg.norm(ref)
    assert err < (30 if eps >= 1e-6 else 10) * eps, (L, loc.shape, err)


@pytest.mark.parametrize("spin", [0, 2])
@pytest.mark.parametrize("eps,sigma", [(1e-5, 1.25), (1e-6, 1.25), (1e-7, 1.25), (1e-8, 1.25), (5e-7, 2.0), (1e-10, 2.0)])
def test_points_per_tile(eps, sigma, spin):
    rng = np.random.default_rng(1700 + spin)
    L = 15
    for n in COUNTS:
        c = np.array([1.2, 2.3])  # one spot, narrower than a tile
        loc = c + rng.uniform(-0.02, 0.02, (n, 2))
        edge = np.array([[0.0, 0.0], [np.pi, 1.0], [1e-3, 6.28], [np.pi - 1e-3, 0.01], [0.7, 2 * np.pi - 1e-9]])
        _run(L, eps, sigma, np.ascontiguousarray(np.concatenate([loc, edge])), rng, spin)


@pytest.mark.parametrize("L", [2, 3, 5])
def test_grid_narrower_than_a_tile(L):
    rng = np.random.default_rng(L)
    loc = np.stack([np.arccos(rng.uniform(-1, 1, 300)), rng.uniform(0, 2 * np.pi, 300)], 1)
    _run(L, 1e-10, 2.0, loc, rng, 2)

"""The kernel polynomials of the interpolation against the exact ES kernel.

psi's polynomial is least exact in the two outer cells of the footprint (branch point at |z| = 1), by eight digits at
epsilon 1e-7.  Points whose offsets are the interpolation nodes of the degree-24 fit, u = cos(pi (j + 1/2) / 25) / 2, see
the outer cells exact and show the other cells alone, which the wide fine grids of these plans need at full accuracy.

Tolerance, relative to the largest value: weights rounded to 2e-16 on both axes, grid values up to about 20 times the
result (the deconvolution at the band limit), sums of 64 to 100 terms: 1e-13."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import almutil, clib, nufft, pipeline

pytestmark = pytest.mark.gpu


def exact_kernel_reference(alm, L, nf, w, beta, theta, phi):
    """The plan's nuFFT (its fine grid, width and beta) with psi itself, from the oracle's parts."""
    sh = pipeline.NuSHT(L)
    cmap = pipeline.phi_synth(clib.sht_synth_rings(alm, L, 0, sh.thetas), L, 0, sh.nphi)
    F = np.fft.fft2(sh._doubling(cmap, 0))
    F /= F.size
    k = np.arange(-L, L + 1)
    grid = np.zeros((nf, nf), dtype=np.complex128)
    d = nufft.es_fourier(k, nf, w, beta)
    grid[np.ix_(k % nf, k % nf)] = F[np.ix_(k % F.shape[0], k % F.shape[1])] / np.outer(d, d)
    return clib.es_interp(np.fft.ifft2(grid) * nf * nf, theta, phi, w, beta).real


def node_points(nf, w, rng, npts=2000):
    """theta in (0, pi), phi in (0, 2 pi) at footprint offsets u = 1/2 cos(pi (j + 1/2) / 25)."""
    u = 0.5 * np.cos(np.pi * (rng.integers(0, 25, (2, npts)) + 0.5) / 25)
    cell = np.stack([rng.integers(1, nf // 2 - 1, npts), rng.integers(1, nf - 1, npts)])  # first cell + w / 2
    return (cell + 0.5 * (w % 2) - 0.5 - u) * (2 * np.pi / nf)


@pytest.mark.parametrize("L,eps,sigma", [(15, 5e-7, 2.0), (40, 1e-7, 2.0), (100, 1e-8, 2.0), (63, 5e-7, 1.5)])
def test_interior_cells_are_exact(L, eps, sigma):
    from cunusht_amd import _lib
    from cunusht_amd.transformer import NuPlan
    rng = np.random.default_rng(2100 + L)
    a = almutil.random_alm(L, 0, 1, rng)
    pl = NuPlan(L, 0, 1, eps, 2000, sigma=sigma)
    i = pl.info()
    nf, w, beta = i["nfine"], i["kernel_width"], i["beta"]
    theta, phi = node_points(nf, w, rng)
    t, p = torch.as_tensor(theta, device="cuda"), torch.as_tensor(phi, device="cuda")
    pl.set_pts(t, p)
    out = torch.empty(theta.size, dtype=torch.float64, device="cuda")
    at = torch.as_tensor(a[0], device="cuda")
    _lib.call("nusht_nusht2d2", pl._h, ctypes.c_void_p(at.data_ptr()), ctypes.c_void_p(out.data_ptr()), None, None,
              ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    ref = exact_kernel_reference(a, L, nf, w, beta, theta, phi)
    err = np.max(np.abs(out.cpu().numpy() - ref)) / np.max(np.abs(ref))
    assert err < 1e-13, (w, err)

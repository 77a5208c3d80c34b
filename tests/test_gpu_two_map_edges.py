"""Launches of two maps (batches of 2, the last two of a batch of 6), in blocks of 8 waves and (lmax 1150) free ones:
l-ranges around multiples of the chunks and ring counts around multiples of 64 pairs, E + B, E alone and spin 0,
against direct summation.

Tolerance, relative 2-norm: ten times epsilon, as in the other comparisons of nusht2d2 with direct summation."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import almutil, clib

pytestmark = pytest.mark.gpu

EPS = 1e-12


def _direct(alm, L, spin, theta, phi):
    G = clib.sht_synth_rings(alm, L, spin, theta)
    if spin == 0:
        m = np.arange(L + 1)
        return np.real(np.sum(np.where(m == 0, 1, 2)[:, None] * G * np.exp(1j * np.outer(m, phi)), axis=0))
    return np.sum(G * np.exp(1j * np.outer(np.arange(-L, L + 1), phi)), axis=0)


@pytest.mark.parametrize("spin,nc", [(0, 1), (1, 1), (1, 2), (2, 1), (2, 2)])
def test_two_maps(spin, nc):
    from cunusht_amd import _lib
    from cunusht_amd.transformer import NuPlan
    rng = np.random.default_rng(2300 + 10 * spin + nc)
    n = 60
    theta, phi = np.arccos(rng.uniform(-1, 1, n)), rng.uniform(0, 2 * np.pi, n)
    t, f = torch.as_tensor(theta, device="cuda"), torch.as_tensor(phi, device="cuda")
    p = lambda x: ctypes.c_void_p(x.data_ptr())
    # the equiangular grid has good_size(2 lmax + 2) / 2 + 1 rings: 65 pairs from lmax 127 on, 129 at 255, 193 at 383
    for L in (2, 7, 8, 9, 16, 25, 40, 70, 124, 127, 128, 255, 383, 1150):
        a = np.stack([almutil.random_alm(L, spin, nc, rng) for _ in range(2)])
        pl = NuPlan(L, spin, nc, EPS, n, max_maps=2)
        pl.set_pts(t, f)
        at = torch.as_tensor(a, device="cuda")
        out = torch.full((2, 2, n), np.nan, dtype=torch.float64, device="cuda")
        _lib.call("nusht_nusht2d2_batch", pl._h, 2, p(at), 2 * at[0].numel(), p(out[0, 0]),
                  p(out[0, 1]) if spin else None, 2 * n, None,
                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        got = out.cpu().numpy()
        for b in range(2):
            full = a[b] if spin == 0 or nc == 2 else np.stack([a[b][0], np.zeros_like(a[b][0])])
            ref = _direct(full, L, spin, theta, phi)
            g = got[b, 0] if spin == 0 else got[b, 0] + 1j * got[b, 1]
            err = np.linalg.norm(g - ref) / np.linalg.norm(ref)
            assert err < 10 * EPS, (L, b, err)

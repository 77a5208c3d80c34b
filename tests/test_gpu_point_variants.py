"""Exact point synthesis at the sizes where the Legendre kernel changes (spin s: 7 and 8 groups of 64 points, 12 000 and
40 000 waves), both contractions, against the oracle's recursion summed over m.

Tolerance, relative to the largest value: 1e-12 up to lmax 320, above in proportion to the recursion steps."""
import numpy as np
import pytest
import torch

from oracle import almutil, clib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,npts", [(300, 2500), (300, 2561), (1800, 448), (1800, 449), (700, 3640), (700, 3649)])
@pytest.mark.parametrize("spin,nc", [(0, 1), (2, 1), (2, 2)])
def test_point_synthesis(spin, nc, L, npts):
    from cunusht_amd.transformer import PointPlan
    rng = np.random.default_rng(L + npts)
    theta = np.arccos(rng.uniform(-1, 1, npts))
    phi = rng.uniform(0, 2 * np.pi, npts)
    a = almutil.random_alm(L, spin, nc, rng)
    got = PointPlan(L, spin, theta).synthesis(torch.as_tensor(a, device="cuda"), nc,
                                              torch.as_tensor(phi, device="cuda")).cpu().numpy()
    sub = rng.choice(npts, 100, replace=False)
    full = a if spin == 0 or nc == 2 else np.stack([a[0], np.zeros_like(a[0])])
    G = clib.sht_synth_rings(full, L, spin, theta[sub])
    if spin == 0:
        m = np.arange(L + 1)
        ref = np.real(np.sum(np.where(m == 0, 1, 2)[:, None] * G * np.exp(1j * np.outer(m, phi[sub])), axis=0))
        got = got[sub]
    else:
        ref = np.sum(G * np.exp(1j * np.outer(np.arange(-L, L + 1), phi[sub])), axis=0)
        got = got[0][sub] + 1j * got[1][sub]
    assert np.max(np.abs(got - ref)) < 1e-12 * max(1.0, L / 320.0) * np.max(np.abs(ref))

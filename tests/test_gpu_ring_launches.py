"""Ring transforms by the launches a plan splits into: more rings than the one launch of a small plan takes (513), with
every workgroup size and DFT method among them (direct, Rader, Bluestein, split), all lengths above the band and lengths
from 1 on; 512 rings of the same kinds, in one launch; rings of one length shorter than their band, staged and not.

Tolerances, relative to the largest value: 1e-12 up to lmax 320 and in proportion to the recursion steps above,
the bound of the other ring-transform tests."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import almutil, clib, pipeline

pytestmark = pytest.mark.gpu

KINDS = [257, 400, 509, 1000, 1009, 1111, 2039, 2048, 2050, 2111, 3079, 4096, 4158, 4161, 4400, 8191, 8192]
LONG = [n for n in KINDS if n > 1100]


def _mixed(kinds, nring, rng):
    return np.concatenate([kinds, rng.choice(kinds[:6], nring - len(kinds))])


@pytest.mark.parametrize("L,nring,kinds", [(60, 513, KINDS), (60, 512, KINDS), (140, 513, [1, 2, 5, 64, 130, 131] + KINDS),
                                           (500, 513, [1, 3, 256, 600, 983, 1000] + LONG), (500, 200, [1001, 1008, 1013]),
                                           (80, 513, [170, 180, 200]), (2500, 6, [4368]), (2300, 6, [4599]),
                                           (4100, 6, [257]), (700, 520, [1024])])
@pytest.mark.parametrize("spin", [0, 2])
def test_ring_launches(spin, L, nring, kinds):
    from cunusht_amd import _lib
    from cunusht_amd.geometry import Geom
    from cunusht_amd.transformer import RingSHT
    rng = np.random.default_rng(100 * spin + L + nring)
    nph = _mixed(kinds, nring, rng)
    rng.shuffle(nph)
    theta = np.pi * (np.arange(nring) + 0.5) / nring
    phi0 = np.where(np.arange(nring) % 3 == 0, 0.0, rng.uniform(0, 2 * np.pi, nring))
    ofs = np.concatenate([[0], np.cumsum(nph)[:-1]])
    npix = int(nph.sum())
    r = RingSHT(Geom(theta, phi0, nph, ofs, np.ones(nring)), L, spin)
    nc = 1 if spin == 0 else 2
    a = almutil.random_alm(L, spin, nc, rng)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    at = torch.as_tensor(a, device="cuda")
    out = torch.full((2, npix), np.nan, dtype=torch.float64, device="cuda")
    _lib.call("nusht_ringplan_synthesis", r._h, p(at), nc, p(out[0]), p(out[1]) if spin else None, st)
    got = out.cpu().numpy()
    got = got[0] if spin == 0 else got[0] + 1j * got[1]
    tol = 1e-12 * max(1.0, L / 320.0)
    G = clib.sht_synth_rings(a, L, spin, theta)
    ref = np.concatenate([pipeline.phi_synth(G[:, i:i + 1], L, spin, int(nph[i]), phi0[i:i + 1]).reshape(-1)
                          for i in range(nring)])
    assert np.max(np.abs(got - ref)) < tol * np.max(np.abs(ref))

    x = rng.standard_normal((2, npix))
    if spin == 0:
        x[1] = 0
    xm = x[0] if spin == 0 else x[0] + 1j * x[1]
    Gt = np.concatenate([pipeline.phi_adjoint(xm[ofs[i]:ofs[i] + nph[i]][None], L, spin, phi0[i:i + 1])
                         for i in range(nring)], axis=1)
    xt = torch.as_tensor(x, device="cuda")
    res = torch.full((nc, (L + 1) * (L + 2) // 2), np.nan, dtype=torch.complex128, device="cuda")
    _lib.call("nusht_ringplan_adjoint", r._h, p(xt[0]), p(xt[1]) if spin else None, p(res), nc, st)
    ref = clib.sht_adjoint_rings(Gt, L, spin, nc, theta)
    assert np.max(np.abs(res.cpu().numpy() - ref)) < tol * np.max(np.abs(ref))

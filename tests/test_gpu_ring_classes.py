"""Ring transforms at the edges of their workgroup sizes and of the sums over aliased rows: rings of 1 to 5 pixels,
lengths around the workgroup sizes, half of them and the 2048 and 4160 values a class holds, smooth, prime and
other lengths mixed in one plan, rows that fit LDS and (lmax 4200, spin 1) rows that do not; theta and phi
transforms of the point-set calls around 2048 and 5120 values.

Tolerances, relative to the largest value: 1e-12 up to lmax 320 and in proportion to the recursion steps above,
the bound of the Legendre tests, for the ring transforms; the requested accuracy for the point sets."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import almutil, clib, pipeline

pytestmark = pytest.mark.gpu


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda")


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


SHORT = [1, 2, 3, 4, 5, 7, 16, 64, 127, 128, 129, 130, 255, 256, 257, 258, 383, 384, 385, 511, 512, 513]
LONG = [767, 768, 769, 1023, 1024, 1025, 1536, 2047, 2048, 2049, 2053, 2054, 4098, 4160, 4161, 4200]


@pytest.mark.parametrize("L,nph", [(30, SHORT), (1020, SHORT + LONG), (1030, SHORT + LONG), (2100, SHORT + LONG),
                                   (1020, [2041]), (1023, [2048]), (1024, [2049]), (2079, [4160]), (2080, [4161]),
                                   (1020, [64, 64]), (4200, [1, 3, 4, 200, 257, 8191])])
@pytest.mark.parametrize("spin", [0, 1, 2])
def test_ring_lengths(spin, L, nph):
    from cunusht_amd import _lib
    from cunusht_amd.geometry import Geom
    from cunusht_amd.transformer import RingSHT
    rng = np.random.default_rng(1000 * spin + L + len(nph))
    nph = np.array(nph)
    nring, npix = len(nph), int(nph.sum())
    theta = np.pi * (np.arange(nring) + 0.5) / nring
    phi0 = np.where(np.arange(nring) % 3 == 0, 0.0, rng.uniform(0, 2 * np.pi, nring))
    ofs = np.concatenate([[0], np.cumsum(nph)[:-1]])
    r = RingSHT(Geom(theta, phi0, nph, ofs, np.ones(nring)), L, spin)
    nc = 1 if spin == 0 else 2
    a = almutil.random_alm(L, spin, nc, rng)
    out = torch.zeros((2, npix), dtype=torch.float64, device="cuda")
    at = _t(a)
    _lib.call("nusht_ringplan_synthesis", r._h, _p(at), nc, _p(out[0]), _p(out[1]) if spin else None, _stream())
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
    xt = _t(x)
    xm = x[0] if spin == 0 else x[0] + 1j * x[1]
    Gt = np.concatenate([pipeline.phi_adjoint(xm[ofs[i]:ofs[i] + nph[i]][None], L, spin, phi0[i:i + 1])
                         for i in range(nring)], axis=1)
    res = torch.zeros((nc, (L + 1) * (L + 2) // 2), dtype=torch.complex128, device="cuda")
    _lib.call("nusht_ringplan_adjoint", r._h, _p(xt[0]), _p(xt[1]) if spin else None, _p(res), nc, _stream())
    ref = clib.sht_adjoint_rings(Gt, L, spin, nc, theta)
    assert np.max(np.abs(res.cpu().numpy() - ref)) < tol * np.max(np.abs(ref))


@pytest.mark.parametrize("L,eps", [(511, 1e-10), (513, 1e-10), (1023, 1e-10), (1025, 1e-10), (1279, 1e-10), (1282, 1e-10),
                                   (2558, 1e-10), (2562, 1e-10), (818, 1e-5), (821, 1e-5), (2047, 1e-5), (2050, 1e-5),
                                   (4095, 1e-5), (4099, 1e-5)])
@pytest.mark.parametrize("spin", [0, 2])
def test_point_set_transform_lengths(spin, L, eps):
    """Fine grids and theta rings with lengths on both sides of 2048, 5120 and 10240, against the ring transform."""
    import cunusht_amd
    from cunusht_amd import _lib
    from cunusht_amd.geometry import Geom
    from cunusht_amd.transformer import RingSHT
    rng = np.random.default_rng(L + spin)
    nring, n = 24, 64
    theta = np.pi * (np.arange(nring) + 0.3) / nring
    phi0 = rng.uniform(0, 2 * np.pi / n, nring)
    r = RingSHT(Geom(theta, phi0, np.full(nring, n), np.arange(nring) * n, np.ones(nring)), L, spin)
    nc = 1 if spin == 0 else 2
    a = almutil.random_alm(L, spin, nc, rng)
    at = _t(a)
    ref = torch.zeros((2, nring * n), dtype=torch.float64, device="cuda")
    _lib.call("nusht_ringplan_synthesis", r._h, _p(at), nc, _p(ref[0]), _p(ref[1]) if spin else None, _stream())
    ref = ref.cpu().numpy()[:nc]
    loc = _t(np.stack([np.repeat(theta, n), (phi0[:, None] + 2 * np.pi * np.arange(n) / n).reshape(-1)], 1))
    x = rng.standard_normal((nc, nring * n))
    T = cunusht_amd.get_transformer("GPU")(("gl", {"lmax": L}), nuFFTtype=2, epsilon=eps, spin=spin)
    y = T.nusht2d2(L, L, _t(a[0] if spin == 0 else a), loc, spin=spin).cpu().numpy().reshape(nc, -1)
    assert np.linalg.norm(y - ref) < 10 * eps * np.linalg.norm(ref)
    ad = T.nusht2d1(L, L, _t(x[0] if spin == 0 else x), loc, spin=spin).cpu().numpy().reshape(nc, -1)
    lhs = float(np.sum(x * ref))
    rhs = sum(almutil.myalmdot(a[c], ad[c], L) for c in range(nc))
    assert abs(lhs - rhs) < 10 * eps * np.linalg.norm(x) * np.linalg.norm(ref)

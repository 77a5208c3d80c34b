"""Legendre kernels at the edges of their loops: l-ranges around multiples of the 2, 4 and 8 l chunks and the
prefetch depth, ring counts around multiples of the 64-pair groups a wave takes (1, 2 or 3 of them), every
synthesis variant, E + B and E only, against the oracle's ring transforms.

Tolerances, relative to the largest value: 1e-12 up to lmax 320, the bound of the other ring-transform tests
there; above, in proportion to the number of recursion steps."""
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


def _ring_plan(L, spin, nring):
    from cunusht_amd.geometry import Geom
    from cunusht_amd.transformer import RingSHT
    nphi = 2 * L + 2
    theta = np.pi * (np.arange(nring) + 0.5) / nring  # mirrored pairs, and an equator ring for odd counts
    geom = Geom(theta, np.zeros(nring), np.full(nring, nphi), np.arange(nring) * nphi, np.ones(nring))
    return RingSHT(geom, L, spin), theta, nphi


@pytest.mark.parametrize("nring", [1, 130, 386])
@pytest.mark.parametrize("spin", [0, 1, 2])
def test_synthesis_chunk_and_group_edges(spin, nring, monkeypatch):
    from cunusht_amd import _lib
    rng = np.random.default_rng(50 + spin + nring)
    for L in (2, 7, 8, 9, 16, 25, 40, 70):
        for nc in (1,) if spin == 0 else (1, 2):
            a = almutil.random_alm(L, spin, nc, rng)
            full = a if spin == 0 or nc == 2 else np.stack([a[0], np.zeros_like(a[0])])
            ref = None
            for v in range(_lib.load().nusht_legendre_variants()):
                monkeypatch.setenv("NUSHT_LEGENDRE_VARIANT", str(v))
                r, theta, nphi = _ring_plan(L, spin, nring)
                out = torch.zeros((2, nring * nphi), dtype=torch.float64, device="cuda")
                at = _t(a)
                _lib.call("nusht_ringplan_synthesis", r._h, _p(at), nc, _p(out[0]), _p(out[1]) if spin else None,
                          _stream())
                got = out.cpu().numpy()
                got = got[0] if spin == 0 else got[0] + 1j * got[1]
                if ref is None:
                    G = clib.sht_synth_rings(full, L, spin, theta)
                    ref = pipeline.phi_synth(G, L, spin, nphi, np.zeros(nring)).reshape(-1)
                err = np.max(np.abs(got - ref)) / np.max(np.abs(ref))
                assert err < 1e-12, (L, nc, v, err)


@pytest.mark.parametrize("nring", [1, 130, 386])
@pytest.mark.parametrize("spin", [0, 1, 2])
def test_adjoint_chunk_and_group_edges(spin, nring):
    """The same for the adjoint (both numbers of ring groups per wave: 1300 needs three), E + B and E only."""
    from cunusht_amd import _lib
    rng = np.random.default_rng(80 + spin + nring)
    for L in (2, 7, 8, 9, 16, 25, 40, 70) + ((1300,) if nring == 386 else ()):
        r, theta, nphi = _ring_plan(L, spin, nring)
        x = rng.standard_normal((2, nring * nphi))
        if spin == 0:
            x[1] = 0
        xt = _t(x)
        xm = (x[0] if spin == 0 else x[0] + 1j * x[1]).reshape(nring, nphi)
        Gt = pipeline.phi_adjoint(xm, L, spin, np.zeros(nring))
        for nc in (1,) if spin == 0 else (1, 2):
            res = torch.full((nc, (L + 1) * (L + 2) // 2), np.nan, dtype=torch.complex128, device="cuda")
            _lib.call("nusht_ringplan_adjoint", r._h, _p(xt[0]), _p(xt[1]) if spin else None, _p(res), nc, _stream())
            ref = clib.sht_adjoint_rings(Gt, L, spin, nc, theta)
            err = np.max(np.abs(res.cpu().numpy() - ref)) / np.max(np.abs(ref))
            assert err < 1e-12 * max(1.0, L / 320.0), (L, nc, err)

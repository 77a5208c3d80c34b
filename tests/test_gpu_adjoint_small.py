"""The adjoint of at most 512 ring pairs, whose waves add up in LDS and write every coefficient: lengths around the 8 l
chunks, ring counts around those of one to eight groups and of two groups per wave, polar rings that join late or (lmax
900) never, few rings at an lmax whose sums leave a CU too few waves (1300), E + B and E alone, output
filled with NaN before, against the oracle.  Up to 384 pairs (512 for spin 0) the result repeats bit for bit.

Tolerance, relative to the largest value: 1e-12 up to lmax 320, above in proportion to the recursion steps."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import almutil, clib, pipeline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nring", [1, 2, 127, 128, 130, 512, 514, 1024])
@pytest.mark.parametrize("spin", [0, 1, 2])
def test_adjoint_in_one_workgroup(spin, nring):
    from cunusht_amd import _lib
    from cunusht_amd.geometry import Geom
    from cunusht_amd.transformer import RingSHT
    rng = np.random.default_rng(2500 + 10 * spin + nring)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for L in (2, 3, 7, 8, 9, 10, 15, 16, 17, 63, 126, 300, 900) + ((1279, 1300) if nring in (2, 130) else ()):
        for theta in ((np.arange(nring) + 0.5) * np.pi / nring, 1e-3 + 0.05 * (np.arange(nring) + 1) / nring):
            nphi = 24
            r = RingSHT(Geom(theta, np.zeros(nring), np.full(nring, nphi), np.arange(nring) * nphi, np.ones(nring)), L, spin)
            if r.info()["ring_pairs"] > 512:
                continue
            x = rng.standard_normal((2, nring * nphi))
            if spin == 0:
                x[1] = 0
            xt = torch.as_tensor(x, device="cuda")
            xm = (x[0] if spin == 0 else x[0] + 1j * x[1]).reshape(nring, nphi)
            Gt = pipeline.phi_adjoint(xm, L, spin, np.zeros(nring))
            for nc in (1,) if spin == 0 else (1, 2):
                res = [torch.full((nc, (L + 1) * (L + 2) // 2), np.nan, dtype=torch.complex128, device="cuda")
                       for _ in range(2)]
                for q in res:
                    _lib.call("nusht_ringplan_adjoint", r._h, p(xt[0]), p(xt[1]) if spin else None, p(q), nc, st)
                if r.info()["ring_pairs"] <= (512 if spin == 0 else 384):
                    assert torch.equal(torch.view_as_real(res[0]), torch.view_as_real(res[1]))
                ref = clib.sht_adjoint_rings(Gt, L, spin, nc, theta)
                err = np.max(np.abs(res[0].cpu().numpy() - ref)) / np.max(np.abs(ref))
                assert err < 1e-12 * max(1.0, L / 320.0), (L, nc, theta[0], err)

"""The ring adjoint repeats bit for bit as long as at most two waves add to one coefficient: up to 384 ring pairs for
spin s and 512 for spin 0 (a Gauss-Legendre grid of lmax 767 or 1023).  Sizes at both ends of every number of ring
groups a wave takes there."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spin,nc,nring", [(0, 1, 256), (0, 1, 258), (0, 1, 768), (0, 1, 1024), (1, 1, 768),
                                           (2, 2, 258), (2, 2, 514), (2, 2, 768), (2, 1, 386)])
def test_adjoint_repeats(spin, nc, nring):
    from cunusht_amd import _lib
    from cunusht_amd.geometry import Geom
    from cunusht_amd.transformer import RingSHT
    L, nphi = nring - 1, 16  # short rings: the adjoint reads nph pixels whatever the band
    theta = np.pi * (np.arange(nring) + 0.5) / nring
    r = RingSHT(Geom(theta, np.zeros(nring), np.full(nring, nphi), np.arange(nring) * nphi, np.ones(nring)), L, spin)
    g = torch.Generator(device="cuda").manual_seed(nring)
    x = torch.randn(2, nring * nphi, dtype=torch.float64, device="cuda", generator=g)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    res = [torch.empty(nc, (L + 1) * (L + 2) // 2, dtype=torch.complex128, device="cuda") for _ in range(2)]
    _lib.call("nusht_ringplan_adjoint", r._h, p(x[0]), p(x[1]) if spin else None, p(res[0]), nc, st)
    for k in range(30):
        _lib.call("nusht_ringplan_adjoint", r._h, p(x[0]), p(x[1]) if spin else None, p(res[1]), nc, st)
        assert torch.equal(torch.view_as_real(res[0]), torch.view_as_real(res[1])), k

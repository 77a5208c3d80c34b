"""The matrix-core spreading (kernel widths 8 to 13) against the LDS-atomic spreading on the same points: every first
row and column offset inside its windows of first cells, windows with one to nine points (its groups of four are padded),
a tile that takes several passes, both poles and the longitude seam.

Tolerance, relative to the largest coefficient: 1e-12 with the FP64 grid (the two kernels sum the same products in
different orders) and 1e-5 with the FP32 grid (its cells are rounded and added in a varying order), as in the other
comparison of the two spreading kernels."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda")


def _plan(L, eps, sigma):
    import cunusht_amd
    return cunusht_amd.get_transformer("GPU")(("gl", {"lmax": L}), nuFFTtype=2, epsilon=eps, spin=2, sigma=sigma)


@pytest.mark.parametrize("eps,sigma,w", [(1e-7, 2.0, 8), (1e-8, 2.0, 9), (1e-9, 2.0, 10), (1e-10, 2.0, 11),
                                         (1e-11, 2.0, 12), (1e-12, 2.0, 13), (2e-5, 1.25, 8), (1e-5, 1.25, 9),
                                         (1e-6, 1.25, 10)])
def test_matrix_core_spreading_windows(eps, sigma, w, monkeypatch):
    L = 63
    rng = np.random.default_rng(900 + w)
    outs = []
    for rows in ("1", "0"):
        monkeypatch.setenv("NUSHT_SPREAD_ROWS", rows)
        T = _plan(L, eps, sigma)
        plan = T._plan_for(2, 2, eps, T.npix())
        info = plan.info()
        assert info["kernel_width"] == w and info["nufft_spread_rows"] == (1 if rows == "1" else 0)
        if not outs:
            h = 2 * np.pi / info["nfine"]
            # one point in each first cell of a 24 x 40 patch, up to nine more in some of them, a dense spot
            r, c = np.meshgrid(np.arange(24), np.arange(40), indexing="ij")
            cells = np.stack([r.ravel(), c.ravel()], 1)
            more = np.repeat(cells[rng.choice(len(cells), 60, replace=False)], rng.integers(1, 10, 60), axis=0)
            spot = np.repeat([[30, 45]], 3000, axis=0)
            cells = np.concatenate([cells, more, spot])
            th = (cells[:, 0] + 8 + rng.uniform(0, 1, len(cells))) * h
            ph = (cells[:, 1] - 7 + rng.uniform(0, 1, len(cells))) * h  # across the seam
            th = np.concatenate([th, [0.0, np.pi, 1e-3, np.pi - 1e-3]])
            ph = np.concatenate([ph, [0.0, 1.0, 6.28, -0.1]])
            x = rng.standard_normal((2, th.size))
            loc, xt = _t(np.stack([th, ph], 1)), _t(x)
        outs.append(T.nusht2d1(L, L, xt, loc, spin=2).cpu().numpy())
        del T, plan
    err = np.max(np.abs(outs[0] - outs[1])) / np.max(np.abs(outs[1]))
    assert err < (1e-12 if eps < 1e-6 else 1e-5), err

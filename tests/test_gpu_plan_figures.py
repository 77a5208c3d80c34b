"""What a plan says of its Legendre synthesis: the chosen variant's measured time, at every size."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spin", [0, 2])
@pytest.mark.parametrize("L", [40, 255, 700])
def test_legendre_ms_is_measured(L, spin):
    from cunusht_amd.geometry import Geom
    from cunusht_amd.transformer import NuPlan, RingSHT
    plan = NuPlan(L, spin, 2 if spin else 1, 1e-7, 100, max_maps=1)
    theta = np.pi * (np.arange(L + 2) + 0.5) / (L + 2)
    nphi = 2 * L + 2
    ring = RingSHT(Geom(theta, np.zeros(L + 2), np.full(L + 2, nphi), np.arange(L + 2) * nphi, np.ones(L + 2)), L, spin)
    for info in (plan.info(), ring.info()):
        assert info["legendre_variant"] >= 0
        assert 1e-3 < info["legendre_ms"] < 1e3, info["legendre_ms"]

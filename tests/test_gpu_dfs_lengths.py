"""Point-set transforms with fine grids on both sides of 2560, the longest that the theta and phi passes give 256 threads
(four workgroups' rows fill the LDS there), and the synthesis kernel that small plans take unmeasured.

Tolerance: that of the comparison at the passes' other lengths, 10 epsilon."""
import pytest

import test_gpu_ring_classes as classes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,eps", [(639, 1e-10), (640, 1e-10), (1023, 1e-7), (1024, 1e-7), (1023, 1e-5), (1024, 1e-5)])
@pytest.mark.parametrize("spin", [0, 2])
def test_fine_grid_lengths(spin, L, eps):
    classes.test_point_set_transform_lengths(spin, L, eps)


@pytest.mark.parametrize("spin", [0, 2])
def test_small_plans_take_row_broadcasts(spin):
    from cunusht_amd.transformer import NuPlan
    plan = NuPlan(64, spin, 1 if spin == 0 else 2, 1e-10, 100)
    assert plan.info()["legendre_variant"] == 0

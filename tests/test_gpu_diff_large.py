"""The differentiable model's contractions in their wide forms, held to the bars of
test_gpu_diff_shapes: two pixels per thread (from 512 blocks on) at every group size of
phases (8, 4, 12, 16) and of seed rows (4, 8, 12, 16), correlation blocks of a whole group of
stretches (from 768 on), and more tap offsets than the staging loops' first pass holds (257),
with one pixel per thread and with two."""
import pytest

from tests import test_gpu_diff_shapes as shapes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_phase,grid,map_res,n_mu,n,vsini,fac", [
    (56, 12, 9, 26, 38000, 2.0, False), (52, 12, 9, 28, 38001, 0.3, False), (60, 12, 9, 20, 52801, 0.2, True),
    (64, 12, 9, 32, 65537, 0.2, False), (5, 30, 16, 3, 4000, 45.0, True), (6, 24, 16, 2, 4100, 104.0, False),
    (4, 12, 9, 2, 262145, 45.0, False)])
def test_wide_forms(n_phase, grid, map_res, n_mu, n, vsini, fac):
    shapes.test_diff_shapes(n_phase, grid, map_res, n_mu, n, vsini, fac)

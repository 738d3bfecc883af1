"""The choice between the two FP64 contractions (plan_grid64): what it reads of the screen radii, which need not ascend nor
end at the largest, and the table form on such screens against the kernel that evaluates every J0.

Tolerance as in test_hankel_grid64_gpu.py: 2.5e-13 of the sum of the absolute terms."""
import numpy as np
import pytest
import torch

from mma_amd import hankel as H
from test_hankel_grid64_gpu import TOL, absolute_terms, case, elementwise, table_bytes

pytestmark = pytest.mark.gpu


def check(src, z, o, r, rho, D, weights, per_plane=False):
    got = H.direct(src, z, o, r, rho, D, weights=None if per_plane else weights, per_plane=per_plane)
    ref = elementwise(src, z, o, r, rho, D, weights, per_plane=per_plane)
    bound = TOL * absolute_terms(src, r, o, weights, per_plane)[:, None, :]
    assert bool(((got - ref).abs() <= bound).all()), float(((got - ref).abs() / bound).max())


SCREENS = {"descending": lambda rho: rho[::-1].copy(),
           "largest inside": lambda rho: np.concatenate([rho[: len(rho) // 2], rho[::-1][: len(rho) - len(rho) // 2]]),
           "largest negative": lambda rho: np.where(np.arange(len(rho)) == 7, -1.3 * rho.max(), rho),
           "ends at zero": lambda rho: np.concatenate([[0.0], rho[1:-1][::-1], [0.0]])}


@pytest.mark.parametrize("screen", sorted(SCREENS))
def test_screens_in_any_order(screen):
    src, z, o, r, rho, D, weights = case(20, 150, 300, 200)
    rho = SCREENS[screen](rho)
    assert table_bytes(src, z, o, r, rho, D, 3, False) > 0
    check(src, z, o, r, rho, D, weights)
    check(src, z, o, r, torch.tensor(rho, device="cuda"), D, weights)  # no copy on the host


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("at", [0, 99, 199])
def test_screens_that_are_not_finite_keep_the_elementwise_kernel(value, at):
    src, z, o, r, rho, D, weights = case(20, 150, 300, 200)
    rho = rho.copy()
    rho[at] = value
    assert table_bytes(src, z, o, r, rho, D, 3, False) == 0


def test_one_radius_beyond_the_grid_keeps_the_elementwise_kernel():
    src, z, o, r, rho, D, weights = case(20, 150, 300, 200)
    for at in (0, 100, 199):
        far = rho.copy()
        far[at] = 400 * rho.max()
        assert table_bytes(src, z, o, r, far, D, 3, False) == 0


# a launch has 65535 rows of blocks at most
@pytest.mark.parametrize("nrho", [65535, 65536, 70001])
def test_more_screen_radii_than_rows_of_a_launch(nrho):
    src, z, o, r, rho, D, weights = case(20, 3, 64, 2)
    rho = np.linspace(0.0, rho.max() / 20, nrho)
    assert table_bytes(src, z, o, r, rho, D, 3, False) > 0
    check(src, z, o, r, rho, D, weights)

"""The FP64 and the split contractions on the far-field workload at full size (256 planes, 512 radii, 1024 screen radii),
against the kernel that evaluates J0 for every element, which shares neither the grid in K r / D nor its
interpolation with them.  Two groups of neighbouring frequencies and single ones in between, so that column tiles of the
product are full, part filled and far apart in frequency.

Tolerances.  The argument K r rho / D of J0 reaches 675, and the three products that form it round it by 3 * 2^-53 of
that; the interpolation adds 2e-16 of an element ('fp64') and GRID_TOL ('fp64-grid'): together below 2.5e-13 and
GRID_TOL + 2.5e-13 of the sum of the absolute terms.  The others keep the bounds of test_hankel_gpu.py, on
max |d| / max |ref|."""
import numpy as np
import pytest
import torch

from mma_amd import hankel as H, workloads as W
from test_hankel_grid64_gpu import TOL, absolute_terms, elementwise

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def workload():
    z, r, o, rho, src, D = W.hankel_workload()
    pick = np.concatenate([np.arange(0, 70), np.arange(100, 2000, 95), np.arange(1985, 2048)])
    z, o, src = z[:-1], o[pick], src[:, pick].contiguous()
    g = torch.Generator().manual_seed(3)
    pre = torch.exp(6j * torch.rand((len(z), len(o)), generator=g, dtype=torch.float64)).cuda().contiguous()
    weights = np.stack([np.full(len(z), z[1] - z[0]), np.eye(len(z))[0], np.eye(len(z))[-1]])
    ref = elementwise(src, z, o, r, rho, D, weights, pre=pre)
    return (src, z, o, r, rho, D), weights, pre, ref


def test_fp64_forms(workload):
    args, weights, pre, ref = workload
    src, z, o, r = args[:4]
    terms = absolute_terms(src, r, o, weights, False)[:, None, :]
    for name, got, tol in (("fp64", H.direct(*args, weights=weights, pre=pre), TOL),
                           ("fp64-grid", H.gridded(*args, weights, pre=pre, kind="fp64-grid"), H.GRID_TOL + TOL)):
        e = float(((got - ref).abs() / terms).max())
        print("%s: %.2e of the absolute terms, %.2e of the largest" % (
            name, e, float((got - ref).abs().max() / ref.abs().max())), flush=True)
        assert e <= tol, name


@pytest.mark.parametrize("kind,tol", [("fp32-mfma", 1e-6), ("bf16x6-mfma", 1e-6), ("fp16x3-mfma", 1e-6),
                                      ("bf16x3-mfma", 2e-6)])
def test_split_forms(workload, kind, tol):
    args, weights, pre, ref = workload
    got = H.gridded(*args, weights, pre=pre, kind=kind)
    for q in range(3):
        e = float((got[q] - ref[q]).abs().max() / ref[q].abs().max())
        print("%s output %d: %.2e" % (kind, q, e), flush=True)
        assert e <= tol

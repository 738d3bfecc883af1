"""The resident TDSE kernels at the grids where one cover ends and the next begins (16 points a lane to 8177, 24 to 12265, 32
to 16353, then several windows; one wave of 16 to 1009, one of 32 in seven waves to 14305), alone and as members of a
lattice that start as far into a lane as they can; several windows with the scan's fourth level (carries that reach beyond
8 lanes); and snapshots of a grid of several windows in one workgroup.

Tolerance as in test_tdse_resident_gpu.py: 40 eps a step at dt / dx^2 = 25, in proportion at 100."""

import numpy as np
import pytest
import torch

from conftest import golden, rel_err
from mma_amd import tdse, workloads as W
from test_tdse_gpu import run_case
from test_tdse_resident_gpu import ATOL, SHAPE, fields

pytestmark = pytest.mark.gpu
EDGES = [1009, 1010, 8177, 8178, 12265, 12266, 14305, 14306, 16353, 16354]


def agree(got, ref, tol):
    got, ref = (np.asarray(v.cpu())[..., :4, :] for v in (got, ref))
    assert np.isfinite(ref).all()
    assert (np.abs(got - ref) <= tol).all(), np.abs(got - ref).max(axis=-1)


def create(num_r, dx=0.1):
    return tdse.Geometry.create_many(num_r, dx, 0.25, W.GRID["a"], W.GRID["e_guess"], W.UNEVEN_CV, 2.0)


@pytest.mark.parametrize("nx", EDGES)
def test_edges_alone(nx):
    geo, dev = create([nx - 1])[0], fields()
    ref = tdse.BatchPlan(geo, dev, config=SHAPE).enqueue()
    agree(tdse.propagate_batch(geo, dev), ref, ATOL)
    agree(tdse.propagate_one(geo, dev[0].contiguous()), ref[0], ATOL)


# a member 2 * lead points smaller than the widest grid starts `lead` points into that one's table
@pytest.mark.parametrize("nx,lanes_of", [(1009, 16), (8177, 16), (12265, 24), (14305, 32), (16353, 32), (16354, 24)])
def test_edges_with_the_largest_lead(nx, lanes_of):
    geos, dev = create([nx - 1, nx - 1 + 2 * (lanes_of - 1)]), fields()
    ref = tdse.BatchPlan(geos, dev, config=SHAPE).enqueue()
    agree(tdse.propagate_batch(geos, dev), ref, ATOL)
    agree(tdse.propagate_one(geos[0], dev[0].contiguous()), ref[0], ATOL)


@pytest.mark.parametrize("nx", [16353, 20001, 33001])
def test_deep_scans(nx):
    geos, dev = create([nx - 1, nx - 1 + 46], dx=0.05), fields()
    assert geos[0].halo_points > 256  # 24 and 32 points a lane, more than 8 of them
    ref = tdse.BatchPlan(geos, dev, config=SHAPE).enqueue()
    agree(tdse.propagate_batch(geos, dev), ref, 4 * ATOL)
    agree(tdse.propagate_one(geos[0], dev[0].contiguous()), ref[0], 4 * ATOL)


@pytest.mark.parametrize("tprint", [0.25, 0.75, 5.0])
@pytest.mark.parametrize("num_r", [17000, 33000])
def test_snapshots_of_several_windows(dll, monkeypatch, num_r, tprint):
    g = dict(golden("ref_short_even.npz"), num_r=num_r, dx=0.1)
    inputs, side = run_case(dll, g, writewft=1, tprint=tprint)
    monkeypatch.setenv("MMA_TDSE_NO_STEP_PARALLEL", "1")
    inputs2, turn = run_case(dll, g, writewft=1, tprint=tprint)
    for k in ("sourceterm", "PopTot", "PopInt", "expval"):
        assert rel_err(getattr(side, "get_" + k)(), getattr(turn, "get_" + k)()) < 1e-12, k
    a, b = side.get_wavefunction(inputs, grids=False), turn.get_wavefunction(inputs2, grids=False)
    assert a.shape == b.shape and a.shape[0] >= 2
    assert max(rel_err(a[r], b[r]) for r in range(len(a))) < 1e-12
    for o, n in ((side, len(a)), (turn, len(b))):
        dll.free_mtrx(o.psi, n)
        o.delete(dll)
    for i in (inputs, inputs2):
        i.delete(dll)


def test_windows_on_a_shared_lattice_match_the_oracle():
    """The library's own launch on members of the uneven workload that share one lattice: the smallest, the widest (31997
    points) and the one with the most work, both in several windows, over 600 steps."""
    from oracle import ctdse as O
    num_r, n_e = W.uneven_work()
    work = (num_r + 1) * (n_e + 2)
    pick = [int(i) for i in np.argsort(work)[:6]] + [int(np.argmax(num_r)), int(np.argmax(work))]
    sel, steps = W.uneven_batch(indices=pick), 600
    geos = create([m["num_r"] for m in sel])
    dev = torch.tensor(np.stack([m["field"][: steps + 1] for m in sel]), device="cuda")
    plan = tdse.BatchPlan(geos, dev)
    assert plan.config.library_choice
    out = plan.replay().cpu().numpy()
    plan.close()
    for i in (0, 6, 7):
        x, psi0 = geos[i].ground_state()
        ref = O.propagate(sel[i]["num_r"], 0.1, W.GRID["a"], 2.0, 0.25, psi0, x, dev[i].cpu().numpy(), steps)
        for r, k in enumerate(("sourceterm", "PopTot", "PopInt", "expval")):
            e = float(np.abs(out[i, r] - ref[k][:steps]).max())
            print(sel[i]["num_r"], k, "%.2e" % e, flush=True)
            assert e <= ATOL[r, 0] * steps / 120, (sel[i]["num_r"], k)

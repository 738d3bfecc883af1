"""The kernel that keeps a state on the chip (tdse_resident.hip), which the library picks by itself,
against the streaming kernel of an explicit launch shape, at the sizes where its cover of a grid changes:
lanes of 16, 24 and 32 points, one to eight waves, part-filled lanes and waves, several windows, grids
that read a shared lattice at an offset, partial runs with saved states, and one instance alone.

Tolerance: both solve the same system with recurrences whose carries are cut at 1e-17, so they differ by
the rounding of a step, below 40 eps relative at dt / dx^2 = 25 (the right-hand side's terms are up to 12.5
times its result, a few of them).  Added up over the 120 steps of a run without cancelling: 120 * 40 * 1.1e-16
= 5.3e-13 of |psi| = 1, on PopTot, PopInt and the dipole (|V'| < 1); on <x> times the |x| <= 100 the packet reaches."""
import numpy as np
import pytest
import torch

from mma_amd import adjoint, tdse, workloads as W

pytestmark = pytest.mark.gpu
STEPS = 120
ATOL = np.array([5.3e-13, 1.1e-12, 1.1e-12, 5.3e-11])[:, None]  # PopTot and PopInt are squares
SHAPE = (4, 3, 1)


def geometry(num_r, psi0=None):
    return tdse.Geometry(num_r, 0.1, 0.25, W.GRID["a"], W.GRID["e_guess"], W.UNEVEN_CV, 2.0, psi0=psi0)


def fields(n=2):
    t = np.arange(STEPS) * 0.25
    f = np.stack([W.sin2_pulse(t, 0.08, W.omega_au(400e-9), 1, phase=0.4 + i) for i in range(n)])
    return torch.tensor(tdse.pad_fields(f), device="cuda")


def agree(got, ref):
    got, ref = (np.asarray(v.cpu())[..., :4, :] for v in (got, ref))
    assert np.isfinite(ref).all()
    assert (np.abs(got - ref) <= ATOL).all(), np.abs(got - ref).max(axis=-1)


# 16 points a lane to 8192, 24 to 12288, 32 to 16384, then windows; one wave ends at 1024 points of 16 a lane
@pytest.mark.parametrize("nx", [61, 1023, 1024, 1025, 1536, 1537, 6145, 8191, 8192, 8193, 12288, 12289, 16384, 16385,
                                33001])
def test_matches_the_streaming_kernel(nx):
    geo, dev = geometry(nx - 1), fields()
    ref = tdse.BatchPlan(geo, dev, config=SHAPE).enqueue()
    agree(tdse.propagate_batch(geo, dev), ref)
    agree(tdse.propagate_one(geo, dev[0].contiguous()), ref[0])


def test_shared_lattice_offsets():
    sizes = [9000, 8998, 8990, 8976, 8002, 3000, 2998, 402, 20000]
    geos = tdse.Geometry.create_many(sizes, 0.1, 0.25, W.GRID["a"], W.GRID["e_guess"], W.UNEVEN_CV, 2.0)
    dev = fields(len(sizes))
    got = tdse.propagate_batch(geos, dev)
    agree(got, tdse.BatchPlan(geos, dev, config=SHAPE).enqueue())
    for i, geo in enumerate(geos):
        agree(tdse.propagate_one(geo, dev[i].contiguous()), got[i])


# 32 points a lane read part of the factor from the lattice's table again in every step, and near a grid's own
# left wall and past its end, where the table is another grid's, from a copy of their own
@pytest.mark.parametrize("sizes", [[16382, 16380, 15000, 14222, 12990], [16001, 13001, 12289], [16382, 20000, 402, 16000]])
def test_shared_lattice_with_32_points(sizes):
    geos = tdse.Geometry.create_many(sizes, 0.1, 0.25, W.GRID["a"], W.GRID["e_guess"], W.UNEVEN_CV, 2.0)
    dev = fields(len(sizes))
    agree(tdse.propagate_batch(geos, dev), tdse.BatchPlan(geos, dev, config=SHAPE).enqueue())


# the ring of observables is written out in halves of 8 steps
@pytest.mark.parametrize("nx", [2001, 9001, 13001, 17001])
@pytest.mark.parametrize("steps", [1, 2, 7, 8, 9, 16, 17, 24, 31])
def test_run_lengths(nx, steps):
    geo, dev = geometry(nx - 1), fields()[:, :steps + 1].contiguous()
    agree(tdse.propagate_batch(geo, dev), tdse.BatchPlan(geo, dev, config=SHAPE).enqueue())


@pytest.mark.parametrize("nx", [2001, 17001])
def test_complex_start_state(nx):
    x, psi = geometry(nx - 1).ground_state()
    geo, dev = geometry(nx - 1, psi * np.exp(0.3j * x)), fields()
    ref = tdse.BatchPlan(geo, dev, config=SHAPE).enqueue()
    agree(tdse.propagate_batch(geo, dev), ref)
    agree(tdse.propagate_one(geo, dev[1].contiguous()), ref[1])


# saves of 7 and 16 steps against blocks of 16, then the rest of the run from a saved state
@pytest.mark.parametrize("nx,every", [(6001, 7), (17001, 7), (17001, 16)])
def test_partial_runs_equal_the_whole(nx, every):
    geo, dev = geometry(nx - 1), fields()
    n = dev.shape[1] - 1
    whole = tdse.propagate_batch(geo, dev)
    F = adjoint.gate(dev)[0].contiguous()
    S, m = adjoint.state_length(geo), n // every
    save = torch.zeros((2, m, S, 2), dtype=torch.float64, device="cuda")
    out = torch.zeros((2, 5, n), dtype=torch.float64, device="cuda")
    adjoint.run_states(geo, F, n, 0, 0, None, save, every, out)
    torch.testing.assert_close(out[:, :4], whole[:, :4], rtol=0, atol=1e-13)
    start = m // 2
    part = torch.zeros_like(out)
    adjoint.run_states(geo, F, n, start * every, 0, save, None, 1, part, init_slot=start - 1)
    k = start * every + 1
    agree(part[:, :, k:], whole[:, :, k:])


# the same with 16, 24 and 32 points a lane and one window, where a run goes on between saves
@pytest.mark.parametrize("nx,every", [(4001, 9), (9001, 8), (13001, 7)])
def test_saves_leave_the_run_alone(nx, every):
    geo, dev = geometry(nx - 1), fields()
    n = dev.shape[1] - 1
    F = adjoint.gate(dev)[0].contiguous()
    save = torch.zeros((2, n // every, adjoint.state_length(geo), 2), dtype=torch.float64, device="cuda")
    out = torch.zeros((2, 5, n), dtype=torch.float64, device="cuda")
    adjoint.run_states(geo, F, n, 0, 0, None, save, every, out)
    assert torch.equal(out[:, :4], tdse.propagate_batch(geo, dev)[:, :4])


def test_given_shape_is_kept_and_the_library_choice_returns():
    geo, dev = geometry(2000), fields()
    plan = tdse.BatchPlan(geo, dev)
    assert plan.config.library_choice and tdse.default_config([geo]).as_tuple() == plan.config.as_tuple()
    again = tdse.BatchPlan(geo, dev, config=plan.config)
    assert again.config.library_choice
    assert torch.equal(plan.enqueue(), again.enqueue())
    fixed = tdse.BatchPlan(geo, dev, config=plan.config.as_tuple())
    assert not fixed.config.library_choice and fixed.config.as_tuple() == plan.config.as_tuple()

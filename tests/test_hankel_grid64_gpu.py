"""The FP64 contraction through one J0 table (hankel_grid64.hip) against the kernel that evaluates J0 for
every element, at the edges of its cover: part-filled blocks of 64 radii, more blocks than a workgroup has waves,
part-filled tiles of the product, planes without weight, every source and pre-factor form; and the calls that
keep the element-wise kernel.

Tolerance: an element's argument x = K r rho / D is below 700, three products round it by 3 * 2^-53 x = 2.4e-13
at most, J0 and the interpolation add less than 1e-15; so the two differ by at most 2.5e-13 of the sum of the absolute
terms (they do by some 1e-15 of it, the roundings being unrelated)."""
from ctypes import byref, c_longlong, c_void_p

import numpy as np
import pytest
import torch

from mma_amd import hankel as H, workloads as W

pytestmark = pytest.mark.gpu
TOL = 2.5e-13


def elementwise(src, z, o, r, rho, D, weights=None, near=True, pre=None, per_plane=False):
    keep = []
    p = H._planes_struct(src, z, o, r, rho, D, near, pre, 0 if pre is None else pre.dim() - 1, keep)
    w = None if per_plane else H._dev(np.atleast_2d(weights))
    n = len(z) if per_plane else w.shape[0]
    out = torch.empty((n, p.nrho, p.no), dtype=torch.complex128, device="cuda")
    H._check(H._L().hk_direct(byref(p), 0 if per_plane else n, H._ptr(w), int(per_plane), H._ptr(out), H._stream()))
    return out


def table_bytes(src, z, o, r, rho, D, n_out, per_plane):
    keep, need = [], c_longlong()
    p = H._planes_struct(src, z, o, r, rho, D, True, None, 0, keep)
    w = torch.zeros((n_out, len(z)), dtype=torch.float64, device="cuda")
    out = torch.empty((len(z) if per_plane else n_out, p.nrho, p.no), dtype=torch.complex128, device="cuda")
    H._check(H._L().hk_direct_work(byref(p), n_out, H._ptr(w), int(per_plane),
                                   c_void_p(np.ascontiguousarray(rho).ctypes.data), H._ptr(out), c_void_p(), byref(need),
                                   H._stream()))
    return need.value


def case(nz, no, nr, nrho, c64=False, seed=0):
    z, r, o, rho, src, D = W.hankel_workload(nz=nz, no=no, nr=nr, nrho=nrho, seed=seed, complex64=c64)
    g = np.random.default_rng(seed)
    weights = g.standard_normal((3, nz)) * 1e-4
    weights[0, nz // 2] = weights[1, : nz // 3] = 0.0
    return src, z[:-1], o, r, rho, D, weights


def absolute_terms(src, r, o, weights, per_plane):
    """Sum of the absolute terms per output and frequency (|J0|, |pre|, |phase| <= 1)."""
    w = np.zeros(len(r))
    w[:-1] += 0.5 * np.diff(r)
    w[1:] += 0.5 * np.diff(r)
    per = (src.abs().to(torch.float64) * torch.tensor(w * r, device="cuda")).sum(-1)  # plane, frequency
    return per if per_plane else torch.tensor(np.abs(weights), device="cuda") @ per


@pytest.mark.parametrize("nz,no,nr,nrho,c64,pre,per_plane", [
    (60, 200, 64, 257, False, 0, False), (60, 193, 65, 300, True, 1, False), (40, 300, 513, 64, False, 2, False),
    (65, 97, 600, 130, False, 1, False), (30, 700, 200, 65, True, 0, True), (12, 333, 1000, 200, False, 1, True)])
def test_matches_the_elementwise_kernel(nz, no, nr, nrho, c64, pre, per_plane):
    src, z, o, r, rho, D, weights = case(nz, no, nr, nrho, c64)
    assert table_bytes(src, z, o, r, rho, D, 3, per_plane) > 0
    factor = None
    if pre:
        g = torch.Generator().manual_seed(1)
        shape = (nz, no) if pre == 1 else (nz, no, nr)
        factor = torch.exp(6j * torch.rand(shape, generator=g, dtype=torch.float64)).cuda().contiguous()
    args = dict(weights=weights, pre=factor, per_plane=per_plane)
    got = H.direct(src, z, o, r, rho, D, near_field=pre != 2, **args)
    ref = elementwise(src, z, o, r, rho, D, near=pre != 2, **args)
    bound = TOL * absolute_terms(src, r, o, weights, per_plane)[:, None, :]
    assert bool(((got - ref).abs() <= bound).all()), float(((got - ref).abs() / bound).max())
    assert torch.equal(got, H.direct(src, z, o, r, rho, D, near_field=pre != 2, **args))  # no order of arrival in the sums


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("plane", [2, 11])  # 11: no output weighs it
def test_values_that_are_not_finite(value, plane):
    src, z, o, r, rho, D, weights = case(20, 150, 300, 200)
    weights[:, 11] = 0.0
    src[plane, 70, 33] = value
    assert table_bytes(src, z, o, r, rho, D, 3, False) > 0
    got = torch.view_as_real(H.direct(src, z, o, r, rho, D, weights=weights))
    assert torch.equal(got.nan_to_num(7.0, 8.0, 9.0),
                       torch.view_as_real(elementwise(src, z, o, r, rho, D, weights)).nan_to_num(7.0, 8.0, 9.0))


def test_calls_that_keep_the_elementwise_kernel():
    src, z, o, r, rho, D, weights = case(20, 150, 300, 200)
    assert table_bytes(src, z, o, r, rho, D, 3, False) > 0
    assert table_bytes(src, z, o, r, 400 * rho, D, 3, False) == 0  # a grid beyond LDS
    assert table_bytes(src, z, o, r, 0 * rho, D, 3, False) == 0
    assert table_bytes(src, z + 1.0, o, r, rho, D, 3, False) == 0  # planes behind the screen
    assert table_bytes(src[:1, :64], z[:1], o[:64], r, rho, D, 3, False) == 0  # too small to pay
    for rr in (r[::-1].copy(), -r):
        assert table_bytes(src, z, o, rr, rho, D, 3, False) == 0
        assert torch.equal(H.direct(src, z, o, rr, rho, D, weights=weights),
                           elementwise(src, z, o, rr, rho, D, weights))


# 16, 16, 8, 2 and 1 parts of the sources; 600 radii are two tiles of them
@pytest.mark.parametrize("nz,no,nr,nrho", [(1, 3, 2, 1), (3, 5, 17, 300), (2, 60, 600, 150), (1, 130, 40, 700),
                                           (1, 300, 40, 900)])
def test_dealt_sources_against_fp64_sums(nz, no, nr, nrho):
    src, z, o, r, rho, D, weights = case(nz, no, nr, nrho)
    got = elementwise(src, z, o, r, rho, D, weights)
    w = np.zeros(nr)
    w[:-1] += 0.5 * np.diff(r)
    w[1:] += 0.5 * np.diff(r)
    K = o / H.C_LIGHT
    ref = np.zeros((3, nrho, no), dtype=complex)
    from scipy.special import j0
    for k in range(nz):
        u = src[k].cpu().numpy() * (w * r) * np.exp(-1j * K[:, None] * r ** 2 / (2 * (D - z[k])))
        J = j0((K / (D - z[k]))[:, None, None] * (rho[:, None] * r))
        ref += weights[:, k, None, None] * np.matmul(J, u[:, :, None])[..., 0].T
    bound = TOL * absolute_terms(src, r, o, weights, False).cpu().numpy()[:, None, :] + 1e-300
    assert (np.abs(got.cpu().numpy() - ref) <= bound).all()

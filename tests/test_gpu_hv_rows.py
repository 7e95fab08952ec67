"""H.v through the fused pass on staged rows at the edges of its layout: rows shorter than, equal to and just past a
wave's 64 columns and past one pass of a block, row counts that leave a partial row group or whole idle blocks,
one, two and four rows per block, uniform and per-bond hopping, several vectors in one call, padded strides.

Against the oracle's operator to 1e-13 of the largest entry (the bound of every H.v path)."""

import ctypes as C

import numpy as np
import pytest
import torch

from oracle import ed_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("ns,nu,nd", [(1, 0, 1), (4, 2, 0), (4, 0, 2), (6, 3, 1), (8, 4, 4), (8, 1, 3), (9, 2, 4),
                                      (10, 5, 5), (11, 3, 5), (13, 6, 3), (13, 4, 6), (14, 2, 7)])
def test_fused_rows_vs_oracle(gpu, ns, nu, nd, uniform):
    from cmpy_amd import SectorHamiltonOperator

    rng = np.random.default_rng(ns * 100 + nu * 10 + nd)
    bonds = [(i, j) for i in range(ns) for j in range(i + 1, ns) if j == i + 1 or rng.random() < 0.3]
    hops = np.full(len(bonds), -0.7) if uniform else rng.uniform(-1, 1, len(bonds))
    eps, u = rng.uniform(-1, 1, ns), rng.uniform(0, 4, ns)
    op = SectorHamiltonOperator(ns, nu, nd, bonds, hops, eps, u, ns)
    ref = O.SectorOperator(ns, nu, nd, bonds, hops, eps, u, ns)
    nvec = 3
    x = rng.standard_normal((nvec, ref.size))
    want = np.stack([ref.matvec(v) for v in x])
    tol = 1e-13 * max(np.abs(want).max(), 1.0)
    got = op.matvec_device(torch.from_numpy(x).cuda()).cpu().numpy()
    assert np.abs(got - want).max() <= tol
    ld = op.num_dn + 3
    xp = np.full((nvec, op.num_up, ld), np.nan)
    xp[:, :, :op.num_dn] = x.reshape(nvec, op.num_up, op.num_dn)
    yp = torch.full((nvec, op.num_up, ld), float("nan"), dtype=torch.float64, device="cuda")
    op.matvec_device_ld(torch.from_numpy(xp).cuda(), ld, out=yp)
    yp = yp.cpu().numpy()
    assert np.all(yp[:, :, op.num_dn:] == 0.0)
    assert np.abs(yp[:, :, :op.num_dn].reshape(nvec, -1) - want).max() <= tol


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("ns,nu,nd", [(6, 3, 2), (8, 4, 4), (13, 5, 3), (12, 6, 6)])
def test_infinities_reach_only_coupled_entries(gpu, ns, nu, nd, uniform):
    """One infinite entry of x, at the first state of a row (what an unused hop slot names), a hop's source and
    elsewhere: y is infinite, with the oracle's sign, exactly where H has an element to it, and finite where it has none."""
    from cmpy_amd import SectorHamiltonOperator

    rng = np.random.default_rng(ns * 10 + nd)
    bonds = [(0, k) for k in range(1, ns)]  # rows of very different length
    hops = np.full(len(bonds), -0.7) if uniform else rng.uniform(0.2, 1, len(bonds))
    eps, u = rng.uniform(-1, 1, ns), rng.uniform(0, 4, ns)
    op = SectorHamiltonOperator(ns, nu, nd, bonds, hops, eps, u, ns)
    ref = O.SectorOperator(ns, nu, nd, bonds, hops, eps, u, ns)
    x = rng.standard_normal(ref.size)
    tol = 1e-13 * np.abs(ref.matvec(x)).max()
    row = int(ref.t_up.indices[ref.t_up.indptr[ref.num_up // 2]])
    for iu, idn in [(0, 0), (row, 0), (ref.num_up - 1, 0), (row, ref.num_dn // 2), (ref.num_up // 2, ref.num_dn - 1)]:
        xi = x.copy()
        xi[iu * ref.num_dn + idn] = np.inf
        want = ref.matvec(xi)
        got = op.matvec(xi)
        assert not np.isnan(want).any() and np.isinf(want).any()
        inf = np.isinf(want)
        assert np.array_equal(got[inf], want[inf])
        assert np.abs(got[~inf] - want[~inf]).max() <= tol


def _rows(op, ld=None, lanczos=0):
    from cmpy_amd import _lib as L

    r = C.c_int32()
    L.call("ed_op_matvec_rows", op.handle, op.num_dn if ld is None else ld, lanczos, C.byref(r))
    return r.value


def _random_model(ns, uniform, density=0.3):
    rng = np.random.default_rng(ns)
    bonds = [(i, j) for i in range(ns) for j in range(i + 1, ns) if j == i + 1 or rng.random() < density]
    hops = np.full(len(bonds), -0.7) if uniform else rng.uniform(-1, 1, len(bonds))
    return bonds, hops, rng.uniform(-1, 1, ns), rng.uniform(0, 4, ns)


def _check_hv(op, ref, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((2, ref.size))
    want = np.stack([ref.matvec(v) for v in x])
    tol = 1e-13 * max(np.abs(want).max(), 1.0)
    assert np.abs(op.matvec_device(torch.from_numpy(x).cuda()).cpu().numpy() - want).max() <= tol
    ld = op.num_dn + 5
    xp = np.full((2, op.num_up, ld), np.nan)
    xp[:, :, :op.num_dn] = x.reshape(2, op.num_up, op.num_dn)
    yp = torch.full((2, op.num_up, ld), float("nan"), dtype=torch.float64, device="cuda")
    op.matvec_device_ld(torch.from_numpy(xp).cuda(), ld, out=yp)
    yp = yp.cpu().numpy()
    assert np.all(yp[:, :, op.num_dn:] == 0.0)
    assert np.abs(yp[:, :, :op.num_dn].reshape(2, -1) - want).max() <= tol


def _check_ground(op, ref):
    """Unreorthogonalised: every step's H.v carries the recurrence's terms (and a beta of its own or a launch for it)."""
    from cmpy_amd import groundstate

    gs, st = groundstate(op, tol=1e-9, reorth=False, return_stats=True)
    assert st.converged
    r = ref.matvec(gs.state) - gs.energy * gs.state
    assert np.linalg.norm(r) <= 2e-9 and abs(np.linalg.norm(gs.state) - 1.0) <= 1e-12
    e = groundstate(op, tol=1e-10, reorth=True).energy
    assert abs(gs.energy - e) <= 1e-9 * max(abs(e), 1.0)


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("ns,nu,nd", [(16, 1, 6), (16, 1, 8), (14, 2, 7), (13, 3, 5)])
def test_few_long_rows_take_columns(gpu, ns, nu, nd, uniform):
    """Few rows of several chunks a wave, and rows past the staging space (12,870 states): the fused pass on columns,
    whose beta is formed by a launch of its own."""
    from cmpy_amd import SectorHamiltonOperator

    args = (ns, nu, nd, *_random_model(ns, uniform, 0.0), ns)
    op, ref = SectorHamiltonOperator(*args), O.SectorOperator(*args)
    assert _rows(op) == _rows(op, op.num_dn + 5) == -1
    _check_hv(op, ref, nu)
    if uniform:
        _check_ground(op, ref)


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("ns,nu,nd", [(16, 3, 5), (14, 7, 7)])
def test_two_passes_for_long_rows_and_large_lanczos_steps(gpu, ns, nu, nd, uniform):
    """Uniform hopping: rows of 4,096 states and more take two passes, and so do the steps, on padded rows, of a Lanczos
    run on the 14-site chain's 11.8 M states, whose single H.v is fused.  Per-bond hopping: all fused."""
    from cmpy_amd import SectorHamiltonOperator, groundstate

    bonds = O.square_bonds(4, 4) if ns == 16 else O.chain_bonds(ns)
    rng = np.random.default_rng(ns)
    hops = np.full(len(bonds), 1.0) if uniform else rng.uniform(0.5, 1, len(bonds))
    op = SectorHamiltonOperator(ns, nu, nd, bonds, hops, np.full(ns, -2.0), np.full(ns, 4.0), ns)
    if ns == 16:
        assert _rows(op) == _rows(op, lanczos=1) == (0 if uniform else 1)
        _check_hv(op, O.SectorOperator(ns, nu, nd, bonds, hops, np.full(ns, -2.0), np.full(ns, 4.0), ns), nu)
        return
    assert _rows(op) == 2 and _rows(op, op.vector_ld, 1) == (0 if uniform else 2)
    assert op.vector_ld == (3440 if uniform else 3432)
    gs = groundstate(op, tol=1e-7, reorth=False, device=True)
    r = op.matvec_device(gs.state) - gs.energy * gs.state
    assert float(torch.linalg.vector_norm(r)) <= 2e-7
    v0 = torch.rand(op.size, dtype=torch.float64, device="cuda") - 0.5
    assert gs.energy <= float(torch.dot(v0, op.matvec_device(v0)) / torch.dot(v0, v0))


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("ns,nu,nd,rows", [(12, 3, 6, 1), (13, 5, 3, 2), (12, 6, 6, 4), (14, 5, 7, 2)])
def test_each_number_of_rows_per_block(gpu, ns, nu, nd, rows, uniform):
    """One, two and four rows a block, with a last block that is not full; the form in a Lanczos step below 10^6 states."""
    from cmpy_amd import SectorHamiltonOperator

    args = (ns, nu, nd, *_random_model(ns, uniform, 0.0), ns)
    op, ref = SectorHamiltonOperator(*args), O.SectorOperator(*args)
    assert _rows(op) == rows
    _check_hv(op, ref, nu)
    if op.size < 10 ** 6:
        assert _rows(op, lanczos=1) == rows
        _check_ground(op, ref)

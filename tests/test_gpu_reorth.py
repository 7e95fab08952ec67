"""Fully reorthogonalised Lanczos steps at the edges of their kernels: sectors below, at and past one 64-state tile,
several tiles per block, and bases past 64, 128 and 256 vectors (where the thread layout and the route change).

The basis is orthonormal to 1e-13 (the bound of full reorthogonalisation) and V^T H V is the tridiagonal of the
returned coefficients to 1e-12 of the spectral scale, with H the oracle's operator."""

import ctypes as C

import numpy as np
import pytest
import torch

from oracle import ed_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns,nu,nd,m", [(2, 1, 1, 4), (3, 1, 2, 9), (5, 2, 2, 100), (5, 2, 3, 65), (6, 3, 3, 300),
                                        (7, 3, 4, 140), (8, 4, 3, 257), (10, 5, 5, 70)])
def test_full_reorthogonalisation_steps(gpu, ns, nu, nd, m):
    from cmpy_amd import SingleImpurityAndersonModel
    from cmpy_amd import _lib as L

    rng = np.random.default_rng(ns)
    eps, v = rng.uniform(-2, 2, ns - 1), rng.uniform(0.2, 1.0, ns - 1)
    model = SingleImpurityAndersonModel(4.0, -2.0, eps, v, mu=0.0, sign_mode="fermion")
    op = model.hamilton_operator(n_up=nu, n_dn=nd)
    D = op.size
    m = min(m, D)
    phi = torch.from_numpy(rng.uniform(-1, 1, D)).cuda()
    nb = C.c_int64()
    L.call("ed_lanczos_coeffs_workspace", op.handle, m, 1, C.byref(nb))
    work = torch.empty(nb.value, dtype=torch.uint8, device="cuda")
    V = torch.zeros((m, D), dtype=torch.float64, device="cuda")
    a, b = np.zeros(m), np.zeros(m)
    n2, steps = C.c_double(), C.c_int32()
    L.call("ed_lanczos_coeffs", op.handle, L.dptr(phi), m, 1, a.ctypes.data_as(C.POINTER(C.c_double)),
           b.ctypes.data_as(C.POINTER(C.c_double)), C.byref(n2), C.byref(steps), L.dptr(V), L.dptr(work), nb.value,
           L.stream_ptr())
    k = steps.value  # fewer than m where the start vector's Krylov space is exhausted
    assert 1 <= k <= m
    V, a, b = V[:k].cpu().numpy(), a[:k], b[:k - 1]
    assert abs(n2.value - float(phi @ phi)) <= 1e-13 * n2.value
    assert np.abs(V @ V.T - np.eye(k)).max() <= 1e-13
    ref = O.siam_operator(nu, nd, 4.0, -2.0, eps, v, 0.0, width=ns)
    T = V @ np.stack([ref.matvec(x) for x in V], axis=1)
    want = np.diag(a) + np.diag(b, 1) + np.diag(b, -1)
    assert np.abs(T - want).max() <= 1e-12 * max(np.abs(want).max(), 1.0)


@pytest.mark.parametrize("ns,nu,nd", [(6, 3, 3), (8, 4, 4)])
@pytest.mark.parametrize("power", [-517, -512, 500])
def test_start_vectors_of_any_length(gpu, ns, nu, nd, power):
    """Fully reorthogonalised steps from a start vector whose length is close to the smallest (its square just below the
    normal numbers, 1 / length squared past the largest) or to the largest with a square: the same ground state."""
    from cmpy_amd import SectorHamiltonOperator, groundstate

    bonds = O.chain_bonds(ns)
    op = SectorHamiltonOperator(ns, nu, nd, bonds, np.ones(len(bonds)), np.full(ns, -2.0), np.full(ns, 4.0), ns)
    v0 = np.random.default_rng(5).uniform(-1, 1, op.size)
    want = groundstate(op, v0=v0, reorth="full")
    got = groundstate(op, v0=np.ldexp(v0, power), reorth="full")
    assert abs(got.energy - want.energy) <= 1e-9 * abs(want.energy)
    assert 1.0 - abs(got.state @ want.state) <= 1e-9

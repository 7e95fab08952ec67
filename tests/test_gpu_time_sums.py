"""The real-time sum over Lanczos coefficients and the time-to-frequency transform at the edges of their kernels.

Time sum: against the eigenpairs of the tridiagonal (numpy).  The expansion has up to 3584 terms of at most 1, each
rounded to 1.1e-16, and the phase (theta - e0) t of up to 4000 carries 4e-13 on either side, so the bound is 2e-12 of
|phi|^2.  Transform: against the oracle to 1e-12 of the largest value (256 partial sums of equal size)."""

import ctypes as C

import numpy as np
import pytest
import torch

from oracle import ed_oracle as O

pytestmark = pytest.mark.gpu


# (m, tmax): one and two entries a thread, a partial last wave, one node, bases past its size (the eigenvector route)
@pytest.mark.parametrize("m,tmax", [(1, 7.0), (2, 30.0), (63, 50.0), (64, 1.0), (129, 200.0), (1100, 900.0),
                                    (2048, 30.0), (2049, 30.0)])
@pytest.mark.parametrize("sign", [1, -1])
def test_tevo_eval(gpu, m, tmax, sign):
    from cmpy_amd import _lib as L

    rng = np.random.default_rng(m)
    a, b = rng.uniform(-2, 2, m), rng.uniform(0.1, 1.0, max(m - 1, 1))
    t = np.concatenate([[0.0, -tmax, tmax, 1e-12, -1e-6], rng.uniform(-tmax, tmax, 60)])
    norm2, e0 = 0.7, -1.3
    td = torch.from_numpy(t).cuda()
    g = torch.full((2 * len(t),), 0.25, dtype=torch.float64, device="cuda")
    dp = C.POINTER(C.c_double)
    for accumulate in (1, 0):
        L.call("ed_tevo_eval", a.ctypes.data_as(dp), b.ctypes.data_as(dp), m, norm2, e0, sign, L.dptr(td), len(t),
               L.dptr(g), accumulate, L.stream_ptr())
        got = g.cpu().numpy().reshape(-1, 2)
        w, v = np.linalg.eigh(np.diag(a) + (np.diag(b[:m - 1], 1) + np.diag(b[:m - 1], -1) if m > 1 else 0.0))
        want = -1j * sign * norm2 * (np.exp(-1j * sign * (w[None, :] - e0) * t[:, None]) @ v[0] ** 2)
        got = got[:, 0] + 1j * got[:, 1] - (0.25 + 0.25j) * accumulate
        assert np.abs(got - want).max() <= 2e-12 * norm2


def _tevo(a, b, norm2, e0, sign, t):
    from cmpy_amd import _lib as L

    dp = C.POINTER(C.c_double)
    td = torch.from_numpy(t).cuda()
    g = torch.full((2 * len(t),), float("nan"), dtype=torch.float64, device="cuda")
    L.call("ed_tevo_eval", a.ctypes.data_as(dp), b.ctypes.data_as(dp), len(a), norm2, e0, sign, L.dptr(td), len(t),
           L.dptr(g), 0, L.stream_ptr())
    g = g.cpu().numpy()
    return g[::2] + 1j * g[1::2]


# the largest number of times the host reads, one more (maxima of blocks), and many; the largest |t| last, first, inside
@pytest.mark.parametrize("nt", [4096, 4097, 300001])
@pytest.mark.parametrize("at", [0, -1, 0.5])
def test_tevo_eval_many_times(gpu, nt, at):
    """The number of terms follows from the largest |t|, wherever it stands.  Bound as above."""
    rng = np.random.default_rng(nt)
    m = 40
    a, b = rng.uniform(-2, 2, m), rng.uniform(0.1, 1.0, m - 1)
    t = rng.uniform(-1, 1, nt)
    k = int(at * nt) if at == 0.5 else at
    t[k] = -90.0
    got = _tevo(a, b, 0.7, -1.3, 1, t)
    assert np.isfinite(got).all()
    pick = np.unique(np.concatenate([[k % nt, 0, nt - 1], rng.integers(0, nt, 50)]))
    w, v = np.linalg.eigh(np.diag(a) + np.diag(b, 1) + np.diag(b, -1))
    want = -0.7j * (np.exp(-1j * (w[None, :] + 1.3) * t[pick, None]) @ v[0] ** 2)
    assert np.abs(got[pick] - want).max() <= 2e-12 * 0.7


@pytest.mark.parametrize("m", [1, 3, 4, 6, 7, 8, 12, 20, 50, 120])
@pytest.mark.parametrize("phase", [1.0, 60.0, 250.0, 1000.0, 3300.0])
def test_tevo_eval_either_side_of_the_rule(gpu, m, phase):
    """Few nodes or long times go to the eigenpairs, many nodes to the terms; both within the bound above."""
    rng = np.random.default_rng(m)
    a, b = rng.uniform(-2, 2, m), rng.uniform(0.1, 1.0, max(m - 1, 1))
    h = np.diag(a) + (np.diag(b[:m - 1], 1) + np.diag(b[:m - 1], -1) if m > 1 else 0.0)
    t = np.append(rng.uniform(-1, 1, 70), 1.0) * phase / max(np.abs(h).sum(axis=1).max(), 1.0)
    got = _tevo(a, b, 0.7, -1.3, -1, t)
    w, v = np.linalg.eigh(h)
    want = 0.7j * (np.exp(1j * (w[None, :] + 1.3) * t[:, None]) @ v[0] ** 2)
    assert np.abs(got - want).max() <= 2e-12 * 0.7


@pytest.mark.parametrize("nt,nz", [(1, 2), (2, 1), (64, 3), (257, 5), (258, 2), (1300, 7)])
def test_fourier_t2z(gpu, nt, nz):
    from cmpy_amd import fourier_t2z

    rng = np.random.default_rng(nt)
    t = np.cumsum(rng.uniform(0.01, 0.4, nt))
    g = rng.standard_normal(nt) + 1j * rng.standard_normal(nt)
    w = rng.uniform(-4, 4, nz)  # |z h| on both sides of the series' range
    z, got = fourier_t2z(t, g, w, eta=0.05)
    want = O.fourier_t2z(t, g, w, eta=0.05)
    want = want[1] if isinstance(want, tuple) else want
    assert np.abs(got - want).max() <= 1e-12 * max(np.abs(want).max(), 1.0)


@pytest.mark.parametrize("nt,nz", [(3, (1 << 24) + 5), (5, 1 << 18), (9, (1 << 18) - 1), (70, 65537), (300, 16385),
                                   (17, 16383), (400, 4095), (3, 1000)])
def test_fourier_t2z_many_frequencies(gpu, nt, nz):
    """One, 4, 16, 64 and 256 threads a frequency, and more frequencies than a launch has room for at 256: the first,
    the last and those around a block's edge against the oracle, as above."""
    from cmpy_amd import _lib as L

    rng = np.random.default_rng(nt)
    t = np.cumsum(rng.uniform(0.01, 0.4, nt))
    g = rng.standard_normal(nt) + 1j * rng.standard_normal(nt)
    at = np.unique([k % nz for k in (0, 1, 3, 4, 63, 64, 255, 256, nz // 2, (1 << 24) - 1, 1 << 24, -257, -2, -1)])
    z = torch.zeros((nz, 2), dtype=torch.float64, device="cuda")
    z[:, 0] = torch.linspace(-4, 4, nz, dtype=torch.float64, device="cuda")
    z[:, 1] = 0.05
    out = torch.full((nz, 2), float("nan"), dtype=torch.float64, device="cuda")
    td = torch.from_numpy(t).cuda()
    gd = torch.from_numpy(np.stack([g.real, g.imag], axis=1).copy()).cuda()
    L.call("ed_fourier_t2z", L.dptr(td), L.dptr(gd), nt, L.dptr(z), nz, L.dptr(out), L.stream_ptr())
    assert not torch.isnan(out).any()
    idx = torch.from_numpy(at).cuda()
    got = out[idx].cpu().numpy()
    want = O.fourier_t2z(t, g, z[idx, 0].cpu().numpy(), eta=0.05)
    want = want[1] if isinstance(want, tuple) else want
    assert np.abs(got[:, 0] + 1j * got[:, 1] - want).max() <= 1e-12 * max(np.abs(want).max(), 1.0)

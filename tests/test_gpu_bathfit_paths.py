"""Routes of the bath-fit backward at the sizes where they change.

Conjugate gradients run on chip for sectors of up to 5,120 states whose hop
lists fit in LDS and through memory otherwise; the per-bond sums take eight
bonds a pass, a Krylov index a lane, device-wide or in one workgroup a model.
The same gradient comes out of each: device-wide and one-workgroup sums differ
only in the order of sums (1e-10 of the largest entry); a batch solved and
differentiated without LDS staging is a separate ground state to a Ritz residual
of 1e-12, within the 1e-6 bar of the dense reference, which the smallest sectors
are also compared with.
"""
import numpy as np
import pytest

from oracle import ed_oracle as O
from test_gpu_bathfit import _check, _loss_grads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "nb,n_up,n_dn",
    [
        (1, 1, 1),    # 4 states
        (2, 1, 1),    # 9
        (8, 1, 1),    # 81, one full pass of bonds
        (9, 1, 2),    # 450, one bond in the second pass
        (15, 1, 1),   # 256, 15 bonds
        (6, 3, 3),    # 1,225, more states than threads
        (7, 4, 4),    # 4,900, on chip
        (12, 2, 2),   # 6,084, through memory
    ],
)
def test_backward_routes_agree(gpu, monkeypatch, nb, n_up, n_dn):
    from cmpy_amd.batch import AndersonBatch, matsubara

    rng = np.random.default_rng(29)
    M = 2
    u = np.full(M, 3.0)
    eb, v = rng.uniform(-3, 3, (M, nb)), rng.uniform(0.1, 1.2, (M, nb))
    wn = matsubara(50.0, 70)
    target = 1.0 / (1j * wn - rng.uniform(-1, 1, (M, 1)))
    kw = dict(u=u, eps_imp=-u / 2, eps_bath=list(eb), v=list(v), mu=0.0, n_up=np.full(M, n_up),
              n_dn=np.full(M, n_dn), keep_basis=True, tol=1e-12, cf_tol=1e-14)

    def grads():
        b = AndersonBatch(**kw)
        _, gr, gi, _ = _loss_grads(b, wn, target)
        return b, gr, gi, np.concatenate(b.backward(gr, gi)[:2], axis=1)

    b, gr, gi, got = grads()
    monkeypatch.setenv("CMPY_AMD_BWD_SPLIT_M", "100000")
    one = np.concatenate(b.backward(gr, gi)[:2], axis=1)
    monkeypatch.delenv("CMPY_AMD_BWD_SPLIT_M")
    assert np.abs(got - one).max() <= 1e-10 * np.abs(one).max()
    monkeypatch.setenv("CMPY_AMD_BATCH_STAGED", "0")
    _check(got, grads()[3], "unstaged")
    monkeypatch.delenv("CMPY_AMD_BATCH_STAGED")
    if nb <= 2:
        for i in range(M):
            _, de, dv = O.bathfit_grad_dense(3.0, -1.5, eb[i], v[i], 0.0, n_up, n_dn, wn, target[i], 0)
            _check(got[i:i + 1], np.concatenate([de, dv])[None], "dense")


def test_number_of_frequencies_changes_on_one_batch(gpu):
    """One batch solved and differentiated at 16, 300 and 16 frequencies: the gradients of fresh batches, and gradients
    of another size than the last solve's G are refused."""
    from cmpy_amd.batch import AndersonBatch, matsubara

    rng = np.random.default_rng(31)
    M, nb = 3, 4
    kw = dict(u=np.full(M, 3.0), eps_imp=-1.5, eps_bath=list(rng.uniform(-3, 3, (M, nb))),
              v=list(rng.uniform(0.1, 1.2, (M, nb))), mu=0.0, keep_basis=True)

    def grads(b, n):
        wn = matsubara(50.0, n)
        _, gr, gi, _ = _loss_grads(b, wn, 1.0 / (1j * wn - np.linspace(-1, 1, M)[:, None]))
        return gr, gi, np.concatenate(b.backward(gr, gi)[:2], axis=1)

    b = AndersonBatch(**kw)
    b.config(-1, 4, 0)
    for n in (16, 300, 16):
        f = AndersonBatch(**kw)
        f.config(-1, 4, 0)
        gr, gi, got = grads(b, n)
        assert np.array_equal(got, grads(f, n)[2])
        with pytest.raises(ValueError, match="last solve"):
            b.backward(gr[:, 1:], gi[:, 1:])
        with pytest.raises(ValueError, match="last solve"):
            b.backward(gr, gi[:, 1:])

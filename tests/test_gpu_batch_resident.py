"""Batched solves of sectors whose vectors stay on chip in block mode.

A workgroup keeps a sector of up to 4,904 states in LDS and registers; larger
ones go through memory.  The sizes lie on both sides of that limit and of the
workgroup's 768 and 1,024 threads, down to a single state, with up to 15 bath
sites (many hops a state).  Block mode is compared with wave mode (which keeps
every vector in memory), and with the oracle where its dense sum is affordable.
Bars: E0 within 1e-10 relative and G within 1e-8 of max |G|; both modes stop
at a Ritz residual of 1e-10, whose square over the gap bounds E0's error.
"""
import numpy as np
import pytest

from test_gpu_batch import _batch, _check, _oracle_model

pytestmark = pytest.mark.gpu

# (bath sites, n_up, n_dn): sector dimension
SECTORS = [
    (1, 0, 0),    # 1
    (1, 1, 1),    # 4
    (2, 1, 2),    # 9
    (5, 3, 3),    # 400
    (6, 2, 3),    # 735, below 768
    (6, 3, 2),    # 735, rows of 21
    (7, 2, 2),    # 784, above 768
    (6, 3, 3),    # 1,225, above 1,024
    (15, 1, 2),   # 1,920, 15 hops a state
    (12, 1, 3),   # 3,718
    (7, 4, 4),    # 4,900, the largest half-filled sector held on chip
    (13, 1, 3),   # 5,096, above the limit
    (12, 2, 2),   # 6,084, above the limit
]


@pytest.mark.parametrize("sign_mode", ["reference", "fermion"])
def test_block_mode_matches_wave_mode_around_the_on_chip_limit(gpu, sign_mode):
    from cmpy_amd.batch import matsubara

    rng = np.random.default_rng(17)
    m = len(SECTORS)
    u = rng.uniform(1.0, 4.0, m)
    eb = [rng.uniform(-2.0, 2.0, nb) for nb, _, _ in SECTORS]
    v = [rng.uniform(0.2, 1.0, nb) for nb, _, _ in SECTORS]
    n_up = np.array([s[1] for s in SECTORS])
    n_dn = np.array([s[2] for s in SECTORS])
    wn = matsubara(50.0, 48)
    kw = dict(u=u, eps_imp=-u / 2, eps_bath=eb, v=v, mu=0.0, n_up=n_up, n_dn=n_dn, sign_mode=sign_mode)
    out = {}
    for mode, shape in (("block", (-1, 8, 0)), ("wave", (1 << 40, 2, 2))):
        b = _batch(**kw)
        b.config(*shape)
        out[mode] = b.solve(wn)
        assert np.all(out[mode].residual <= 1e-9), (mode, out[mode].residual)
    for i, (nb, nu, nd) in enumerate(SECTORS):
        _check(out["block"], out["wave"].e0[i], out["wave"].g[i], i)
        if nb <= 5:
            e0, g = _oracle_model(u[i], -u[i] / 2, eb[i], v[i], 0.0, nu, nd, wn, width=0 if sign_mode == "reference" else nb + 1)
            _check(out["block"], e0, g, i)

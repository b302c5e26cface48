"""Set-up of the wave part: scan of the origin cells' counts over one chunk (L = 10.6: at most 4096 cells), some
(L = 45) and more than a workgroup sums by itself (L = 172: 5.8 million cells, 1424 chunks).

The product does not depend on the grid cell that the spheres are shifted to (by a part of a cell it does, by
the method's own error of 1e-3); a sphere that a wrong start or place loses changes it in the first
digit.  Shifting by half the grid's cells moves every sphere to other cells and
rounds its coordinates anew (2^-24 L against the Gaussian's width 1.5: 1e-5 relative at L = 172); 1e-4 is
allowed.  A second product of a context starts from what the first left and has to equal a fresh one's.

A product whose positions have moved finds that after its wave part is queued, rebuilds the list and sums
real space over the new one: it differs from a fresh context's in the order of the sums only (1e-6;
1e-5 allowed).  So do the lubrication operators.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _pos(p):
    return torch.tensor(np.concatenate([p, np.zeros((len(p), 1))], 1).astype(np.float32), device="cuda")


def _lattice(N, L, rng, jitter):
    n = int(np.ceil(N ** (1 / 3)))
    cell = np.stack(np.meshgrid(*[np.arange(n)] * 3, indexing="ij"), -1).reshape(-1, 3)[:N]
    return (cell + 0.5) * (L / n) - L / 2 + rng.uniform(-jitter, jitter, (N, 3))


@pytest.mark.parametrize("N, L", [(64, 10.6), (1500, 45.0), (700, 172.0)])
def test_origin_cells(N, L):
    from fsd_amd.stokes import Stokes
    rng = np.random.default_rng(N)
    p = _lattice(N, L, rng, 0.1)
    x = torch.tensor(rng.standard_normal(11 * N).astype(np.float32), device="cuda")
    st, fresh = Stokes(N, L), Stokes(N, L)
    n = st.pse_info()["Nx"]
    q = p + n // 2 * L / n
    q -= L * np.floor(q / L + 0.5)
    a, b = _pos(p), _pos(q)
    st.build_nlist(a)
    fresh.build_nlist(a)
    u1, u2, v = st.mobility(a, x, 2), st.mobility(a, x, 2), fresh.mobility(a, x, 2)
    assert torch.equal(u1, u2) and torch.equal(u1, v)
    fresh.build_nlist(b)
    w = fresh.mobility(b, x, 2)
    assert (w - u1).abs().max() <= 1e-4 * u1.abs().max()


@pytest.mark.parametrize("N, L", [(64, 12.0), (1500, 45.0)])      # list over all pairs, over cells
def test_list_rebuilt_in_product(N, L):
    from fsd_amd.stokes import Stokes
    rng = np.random.default_rng(N)
    p = _lattice(N, L, rng, 0.1)
    q = p[rng.permutation(N)]                # every sphere somewhere else
    x = torch.tensor(rng.standard_normal(11 * N).astype(np.float32), device="cuda")
    y = torch.tensor(rng.standard_normal(17 * N).astype(np.float32), device="cuda")
    st, fresh = Stokes(N, L), Stokes(N, L)
    st.build_nlist(_pos(p))
    fresh.build_nlist(_pos(q))
    b = _pos(q)
    for got, want in ((st.mobility(b, x), fresh.mobility(b, x)), (st.mobility(b, x), fresh.mobility(b, x))):
        assert (got - want).abs().max() <= 1e-5 * want.abs().max()
    ops = (lambda s: s.saddle_multiply(b, y), lambda s: s.rfu(b, y[:6 * N]), lambda s: s.rsu(b, y[:6 * N]),
           lambda s: s.rfe(b, 1.0), lambda s: s.rse(b, 1.0))
    for op in ops:                           # the last four run again if the check they are queued behind says so
        st.build_nlist(_pos(p))
        got, want = op(st), op(fresh)
        assert (got - want).abs().max() <= 1e-5 * want.abs().max()

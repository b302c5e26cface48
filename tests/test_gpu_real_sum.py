"""Real-space sum: the kernel with the table in LDS against the one that reads it from global memory.

A periodic box of spheres and its 3 x 3 x 3 copies have the same real-space sums.  The box (fewer
than 0.7 million list entries) takes the table from global memory, its copies from LDS.  Box length
and coordinates are multiples of 2^-12, so every separation is exact in both and the pair terms are
equal: the two differ in the order of their ~80 terms only.  With that many roundings of a running
sum at 2^-24 of it, random in sign, the difference is about 1e-6 of the largest entry; 2e-5 is allowed.

The lanes per particle that the autotuner can choose, where the table is in LDS, against the FP64 oracle
(1e-5, as for every mobility product).
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N, overlap", [(512, False), (512, True), (509, True)])
def test_table_in_lds(N, overlap):
    from fsd_amd.stokes import Stokes
    L, q = 17.0, 4096.0
    rng = np.random.default_rng(N + overlap)
    n = 8
    cell = np.stack(np.meshgrid(*[np.arange(n)] * 3, indexing="ij"), -1).reshape(-1, 3)[:N]
    pos = (cell + 0.5) * (L / n) - L / 2 + rng.uniform(-0.04, 0.04, (N, 3))
    if overlap:                      # pairs below the rows held in LDS, down to almost touching centres
        pos[1] = pos[0] + [0.5, 0.25, 0.0]
        pos[8] = pos[7] + [1.0, 1.0, 1.25]
    pos = np.round(pos * q) / q
    x = rng.standard_normal(11 * N).astype(np.float32)
    out = []
    for rep in (1, 3):
        shift = np.stack(np.meshgrid(*[np.arange(rep) - rep // 2] * 3, indexing="ij"), -1).reshape(-1, 3) * L
        p = (shift[:, None, :] + pos[None]).reshape(-1, 3)
        k = rep ** 3
        gf = np.concatenate([np.tile(x[:6 * N], k), np.tile(x[6 * N:], k)])
        st = Stokes(k * N, rep * L)
        p4 = torch.tensor(np.concatenate([p, np.zeros((k * N, 1))], 1).astype(np.float32), device="cuda")
        st.build_nlist(p4)
        u = st.mobility(p4, torch.tensor(gf, device="cuda"), 1).cpu().numpy().astype(np.float64)
        out.append((u[:6 * k * N].reshape(k, N, 6), u[6 * k * N:].reshape(k, N, 5)))
    for a, b in zip(*out):
        assert np.abs(b - a).max() <= 2e-5 * np.abs(a).max()


@pytest.mark.parametrize("lanes", [4, 8, 16])
@pytest.mark.parametrize("N", [13824, 13823])
def test_lanes_with_table_in_lds(N, lanes):
    from fsd_amd.stokes import Stokes
    from oracle.oracle import Oracle
    n, L = 24, 51.0
    rng = np.random.default_rng(N)
    cell = np.stack(np.meshgrid(*[np.arange(n)] * 3, indexing="ij"), -1).reshape(-1, 3)[:N]
    pos = ((cell + 0.5) * (L / n) - L / 2 + rng.uniform(-0.05, 0.05, (N, 3))).astype(np.float32)
    x = rng.standard_normal(11 * N).astype(np.float32)
    st = Stokes(N, L)
    p4 = torch.tensor(np.concatenate([pos, np.zeros((N, 1), np.float32)], 1), device="cuda")
    st.build_nlist(p4)
    assert st.get_nlist()[0].sum() >= 700000       # from there on the table is in LDS
    st.set_tuning(real_lanes=lanes)
    u = st.mobility(p4, torch.tensor(x, device="cuda"), 1).cpu().numpy().astype(np.float64)
    ref = Oracle(pos, L).mobility(x, 1)
    assert np.abs(u - ref).max() <= 1e-5 * np.abs(ref).max()

"""Neighbour-list scans by 16 lanes per particle at the sizes where they can go
wrong: fewer particles than a group of 16, one more than a workgroup's 16 groups,
lists that do not fill their last chunk of 16, a list built over all pairs, and a
cluster of overlapping spheres (a cell of more than 256 particles, lists and pair
records that outgrow their first capacity).  Neighbour sets are bit-exact against
the FP64 oracle; operators are within 1e-5 relative (sums of at most 300 FP32 terms
of similar size: 300 * 6e-8 = 2e-5 at worst, the square root of it in practice).
"""
import numpy as np
import pytest

from tests._cases import packing, rel_err, random_vec, sorted_lists

pytestmark = pytest.mark.gpu


def _positions(case):
    if case == "cluster":       # 300 centres inside a radius of 2, the others spread over the box
        rng = np.random.default_rng(5)
        v = rng.standard_normal((300, 3))
        v *= (2.0 * rng.uniform(0.2, 1.0, size=(300, 1)) ** (1 / 3)) / np.linalg.norm(v, axis=1, keepdims=True)
        far = rng.uniform(-10.0, 10.0, size=(117, 3))
        return np.concatenate([v + 2.8, far]).astype(np.float32), 20.0
    n, phi, L = case
    pos, L0 = packing(n, phi, 3)
    if L is None or L0 >= L:
        return pos, L0
    return (pos * np.float32(L / L0)).astype(np.float32), L


@pytest.mark.parametrize("case", [(1, 0.01, 11.0), (15, 0.05, 11.0), (17, 0.05, 18.0), (257, 0.2, None),
                                  (300, 0.3, None), "cluster"])
def test_pair_scan(case):
    import torch
    from fsd_amd.stokes import Stokes
    from oracle.oracle import Oracle
    pos, L = _positions(case)
    N = pos.shape[0]
    print("pair scan", case, "N", N, "L", L, flush=True)
    p4 = np.zeros((N, 4), dtype=np.float32)
    p4[:, :3] = pos
    dpos = torch.from_numpy(p4.reshape(-1)).cuda()
    st = Stokes(N, L)
    st.build_nlist(dpos)
    orc = Oracle(pos, L)
    assert sorted_lists(*st.get_nlist()) == sorted_lists(orc.nneigh, orc.nbrs)
    U = random_vec(6 * N, 4).astype(np.float32)
    dU = torch.from_numpy(U).cuda()
    got = {"rfu": st.rfu(dpos, dU), "rfe": st.rfe(dpos, 1.0), "rsu": st.rsu(dpos, dU), "rse": st.rse(dpos, 1.0),
           "force": st.force_law(dpos)}
    ref = {"rfu": orc.rfu(U), "rfe": orc.rfe(1.0), "rsu": orc.rsu(U), "rse": orc.rse(1.0), "force": orc.force_law()}
    for k in got:
        assert rel_err(got[k].cpu().numpy(), ref[k]) < 1e-5, k

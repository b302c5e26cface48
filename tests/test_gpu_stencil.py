"""Spreading and contraction kernels at the edges of their tiles, against the FP64 oracle: a tile
with more spheres than one staged part holds (400 in a corner of the box, across its faces), grids
whose last tile along an axis is partial, rows that are not a multiple of four nodes, positions
handed in above the box, and a tilted box.  1e-5 relative, as for every mobility product."""
import numpy as np
import pytest

from tests._cases import rel_err, random_vec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("points,xy", [(12, 0.0), (15, 0.3), (16, -0.5), (18, 0.0), (27, 0.25)])
@pytest.mark.parametrize("where", ["spread", "corner", "outside"])
def test_stencil_tiles(points, xy, where):
    import torch
    from fsd_amd.stokes import Stokes
    from oracle.oracle import Oracle
    L = max((points - 0.5) * np.pi / 3.0, 10.6)
    rng = np.random.default_rng(points)
    pos = rng.uniform(-0.5, 0.5, size=(500, 3)) * L * 0.999
    if where == "corner":
        pos[:400] = 0.5 * L + rng.uniform(-1.6, 1.6, size=(400, 3))
        pos = (pos + 0.5 * L) % L - 0.5 * L
    pos = pos.astype(np.float32)
    handed = pos.copy()
    if where == "outside":      # up to two periods above the box along z (the tilt does not move them)
        handed[:, 2] += (np.arange(500) % 3).astype(np.float32) * np.float32(L)
    N = len(pos)
    print("stencil tiles", points, xy, where, flush=True)
    p4 = np.zeros((N, 4), dtype=np.float32)
    p4[:, :3] = handed
    st = Stokes(N, (L, L, L, xy, 0.0, 0.0))
    assert st.pse_info()["Nx"] == points
    dpos = torch.from_numpy(p4.reshape(-1)).cuda()
    gF = random_vec(11 * N, 3).astype(np.float32)
    st.build_nlist(dpos)
    got = st.mobility(dpos, torch.from_numpy(gF).cuda(), 2).cpu().numpy()
    ref = Oracle(pos, L, xy=xy).mobility(gF, 2)     # the oracle takes positions inside the box
    assert rel_err(got, ref) < 1e-5

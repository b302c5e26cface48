"""The far field's transforms (k_fft.hip) against the 3-D library transforms and the FP64
oracle, on grids of each kind: lengths of one, two and three radices, odd and even (the
Nyquist planes), an odd number of rows, three different lengths, planes of each workgroup
size, a tilted box; a grid too large for LDS, which the 3-D plans serve; and planes too large
for it with an x axis that is not, which take the library's 2-D plans and the x pass.

Tolerance: two FP32 transforms of length n differ by about log2(n^3) 6e-8 of the result's
norm, and the largest entry is a few norms per entry: 1e-5 relative, as for every operator."""
import numpy as np
import pytest

from tests._cases import rel_err, rel_err2, random_vec

pytestmark = pytest.mark.gpu


def _edge(n):
    """a box edge whose grid has n points (the grid is the next smooth length of 3 L / pi + 1)"""
    return (n - 0.5) * np.pi / 3.0


# N spheres anywhere in the box (the far field needs no packing)
GRIDS = [(12, 15, 16), (20, 20, 20), (25, 25, 25), (27, 24, 30), (75, 16, 125), (72, 72, 72), (96, 90, 81),
         (128, 25, 12), (18, 135, 135), (12, 150, 160), (15, 162, 192)]


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("xy", [0.0, 0.4])
def test_lds_transforms_match_library_and_oracle(grid, xy, monkeypatch):
    import torch
    from fsd_amd.stokes import Stokes
    L = [_edge(n) for n in grid]
    N = 97
    rng = np.random.default_rng(sum(grid))
    pos = rng.uniform(-0.45, 0.45, size=(N, 3)) * np.array(L)
    p4 = np.zeros((N, 4), dtype=np.float32)
    p4[:, :3] = pos
    dpos = torch.from_numpy(p4.reshape(-1)).cuda()
    gF = torch.from_numpy(random_vec(11 * N, 3).astype(np.float32)).cuda()
    print("grid", grid, "xy", xy, flush=True)
    out = {}
    for f3 in ("0", "1"):
        monkeypatch.setenv("FSD_FFT_3D", f3)
        st = Stokes(N, (*L, xy, 0.0, 0.0))
        pse = st.pse_info()
        assert (pse["Nx"], pse["Ny"], pse["Nz"]) == grid
        st.build_nlist(dpos)
        out[f3] = st.mobility(dpos, gF, 2).cpu().numpy()
        # the Brownian slip needs the inverse alone
        st.setT(1.0)
        out[f3 + "b"] = st.brownian_farfield(dpos, 3).cpu().numpy()
    assert rel_err(out["0"], out["1"]) < 1e-5
    assert rel_err2(out["0b"], out["1b"]) < 1e-5
    if len(set(grid)) == 1 and xy == 0.0:
        from oracle.oracle import Oracle
        orc = Oracle(p4[:, :3], L[0])
        assert rel_err(out["0"], orc.mobility(gF.cpu().numpy(), 2)) < 1e-5


def test_grid_beyond_lds_uses_the_library(monkeypatch):
    """planes of 225 x 240 points exceed LDS: the 3-D plans serve them, with the same result"""
    import torch
    from fsd_amd.stokes import Stokes
    L = [_edge(12), _edge(225), _edge(240)]
    N = 33
    pos = np.random.default_rng(1).uniform(-0.45, 0.45, size=(N, 3)) * np.array(L)
    p4 = np.zeros((N, 4), dtype=np.float32)
    p4[:, :3] = pos
    dpos = torch.from_numpy(p4.reshape(-1)).cuda()
    gF = torch.from_numpy(random_vec(11 * N, 3).astype(np.float32)).cuda()
    out = []
    for f3 in ("0", "1"):
        monkeypatch.setenv("FSD_FFT_3D", f3)
        st = Stokes(N, L)
        assert (st.pse_info()["Ny"], st.pse_info()["Nz"]) == (225, 240)
        st.build_nlist(dpos)
        out.append(st.mobility(dpos, gF, 2).cpu().numpy())
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("grid,xy", [((40, 225, 240), 0.4), ((45, 240, 225), 0.0), ((48, 200, 216), 0.0)])
def test_x_pass_of_planes_beyond_lds(grid, xy, monkeypatch):
    """planes beyond LDS do not take the x pass away: the library's 2-D plans and the x pass give what the
    3-D plans do, and the autotuner finds them the faster ones (48 x 200 x 216: 523 and 711 us)"""
    import torch
    from fsd_amd.stokes import Stokes
    L = [_edge(n) for n in grid]
    N = 33
    pos = np.random.default_rng(2).uniform(-0.45, 0.45, size=(N, 3)) * np.array(L)
    p4 = np.zeros((N, 4), dtype=np.float32)
    p4[:, :3] = pos
    dpos = torch.from_numpy(p4.reshape(-1)).cuda()
    gF = torch.from_numpy(random_vec(11 * N, 3).astype(np.float32)).cuda()
    out = {}
    for f3 in ("0", "1"):
        monkeypatch.setenv("FSD_FFT_3D", f3)
        print("grid", grid, "xy", xy, "3-D plans", f3, flush=True)
        st = Stokes(N, (*L, xy, 0.0, 0.0))
        pse = st.pse_info()
        assert (pse["Nx"], pse["Ny"], pse["Nz"]) == grid
        st.build_nlist(dpos)
        out[f3] = st.mobility(dpos, gF, 2).cpu().numpy()
        st.setT(1.0)
        out[f3 + "b"] = st.brownian_farfield(dpos, 3).cpu().numpy()
        if grid[0] == 48:
            assert st.autotune(dpos)[0]["xpass"] == int(f3)
    assert rel_err(out["0"], out["1"]) < 1e-5
    assert rel_err2(out["0b"], out["1b"]) < 1e-5

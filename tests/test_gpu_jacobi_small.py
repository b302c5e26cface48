"""The applications of the folded factor, by one workgroup and by one launch per iteration, and the
limits between them: no contacts at all, fewer entries than groups, rows that cross groups, rows of
more than four entries, the most rows (1900) with the most blocks (2046 of 2048 allowed) and just
beyond either (1901 rows; 2051 and 2722 blocks).  IC(0), as a mode of its own and as what the learned
mode runs without weights, is compared with the oracle's k-step application of the same factor (1e-4,
the factor's own FP32 tolerance) and the saddle form with the plain one (the same g twice: 1e-6).  The
learned factor, with weights, is compared with its 64-bit application on the GPU's own blocks, where
only FP32 rounding remains (1e-5), for odd and even numbers of iterations."""
import numpy as np
import pytest

from tests._cases import packing, rel_err, random_vec

pytestmark = pytest.mark.gpu


def _t(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32).reshape(-1)).cuda()


# lower blocks at the limit of one workgroup (2048) and beyond it
BLOCKS = {(1900, 0.219): 2046, (1900, 0.2195): 2051, (1000, 0.50): 2722}


def one_workgroup(N, phi, k):
    """its limits, and where the iterations are enough to pay for its first and last steps (N = 1900 and k = 1:
    63 us against 41 by launches; 700 and 2: 50 against 47)"""
    return N <= 1900 and BLOCKS.get((N, phi), 0) <= 2048 and (k >= 5 or N <= 300 * k + 50)


@pytest.mark.parametrize("N,phi,k", [(1, 0.01, 3), (40, 0.10, 2), (171, 0.30, 5), (343, 0.45, 8), (700, 0.40, 3),
                                     (1000, 0.50, 3), (1900, 0.12, 4), (1901, 0.12, 4), (1900, 0.219, 5),
                                     (1900, 0.2195, 5), (1901, 0.12, 5), (700, 0.40, 2), (1900, 0.219, 1)])
@pytest.mark.parametrize("mode", ["ichol_jacobi", "learned"])
def test_small_application(N, phi, k, mode):
    import torch
    from fsd_amd.stokes import Stokes
    from oracle.oracle import Oracle
    pos, L = packing(N, phi, 21)
    if L < 11.0:
        pos, L = (pos * np.float32(11.0 / L)).astype(np.float32), 11.0
    print("small application", N, phi, k, mode, flush=True)
    st = Stokes(N, L, precond=mode, jacobi_iters=k, learned_weights=None, fallback_jacobi=k)
    p4 = np.zeros((N, 4), dtype=np.float32)
    p4[:, :3] = pos
    dpos = torch.from_numpy(p4.reshape(-1)).cuda()
    st.build_nlist(dpos)
    info = st.build_precond(dpos)
    if (N, phi) in BLOCKS:
        assert info["lower_blocks"] == BLOCKS[N, phi]
    orc = Oracle(pos, L)
    orc.build_precond()
    x = random_vec(6 * N, 4).astype(np.float32)
    st.profile(True, classes=["jacobi"])
    g = st.precond_apply(_t(x)).cpu().numpy()
    # launches of the forward iterations: none by one workgroup
    assert st.profile_get("jacobi")[0] == (0 if one_workgroup(N, phi, k) else k)
    assert rel_err(g, orc.precond_apply_jacobi(x, k)) < 1e-4
    b = random_vec(17 * N, 5).astype(np.float32)
    d = st.precond_apply(_t(b[:6 * N] - b[11 * N:])).cpu().numpy()
    xs = st.saddle_precond(_t(b)).cpu().numpy()
    ref = np.concatenate([b[:6 * N] - d, b[6 * N:11 * N], d])
    assert rel_err(xs, ref) < 1e-6


@pytest.mark.parametrize("N,phi,k", [(40, 0.10, 2), (343, 0.45, 1), (700, 0.40, 8), (1900, 0.219, 5), (1900, 0.2195, 5),
                                     (1000, 0.50, 4), (1000, 0.50, 3), (1901, 0.12, 2), (2100, 0.30, 5), (2100, 0.30, 1)])
def test_learned_application(N, phi, k):
    from fsd_amd.stokes import Stokes
    from oracle.oracle import Oracle
    from oracle.learned import LearnedOracle, init_weights
    pos, L = packing(N, phi, 21)
    if L < 11.0:
        pos, L = (pos * np.float32(11.0 / L)).astype(np.float32), 11.0
    print("learned application", N, phi, k, flush=True)
    st = Stokes(N, L, precond="learned", jacobi_iters=k, learned_weights=init_weights(1, scale_out=0.3))
    p4 = np.zeros((N, 4), dtype=np.float32)
    p4[:, :3] = pos
    dpos = _t(p4)
    st.build_nlist(dpos)
    info = st.build_precond(dpos)
    assert info["precond_used"] == 1 and info["fallback"] == 0
    orc = Oracle(pos, L)
    orc.build_precond()
    lo = LearnedOracle(orc, k=k)
    f = st.learned_export(lo.E)
    W, Dinv = f["W"].astype(np.float64), f["Dinv"].astype(np.float64)
    x = random_vec(6 * N, 4).astype(np.float32)
    assert rel_err(st.precond_apply(_t(x)).cpu().numpy(), lo.apply_G(W, Dinv, x)) < 1e-5
    b = random_vec(17 * N, 5).astype(np.float32)
    g = lo.apply_G(W, Dinv, b[:6 * N].astype(np.float64) - b[11 * N:])
    ref = np.concatenate([b[:6 * N] - g, b[6 * N:11 * N], g])
    assert rel_err(st.saddle_precond(_t(b)).cpu().numpy(), ref) < 1e-5

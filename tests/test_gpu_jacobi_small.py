"""The one-workgroup application of the folded factor and its limits: no contacts at all, fewer
entries than groups, rows that cross groups, rows of more than four entries, the largest size it
takes and the first beyond (which runs one launch per iteration); each against the oracle's
k-step application of the same IC(0) factor (1e-4, the factor's own FP32 tolerance), and the
saddle form against the plain one (the same g twice: 1e-6)."""
import numpy as np
import pytest

from tests._cases import packing, rel_err, random_vec

pytestmark = pytest.mark.gpu


def _t(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32).reshape(-1)).cuda()


@pytest.mark.parametrize("N,phi,k", [(1, 0.01, 3), (40, 0.10, 2), (171, 0.30, 5), (343, 0.45, 8), (700, 0.40, 3),
                                     (1000, 0.50, 3), (1900, 0.12, 4), (1901, 0.12, 4)])
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
    st.build_precond(dpos)
    orc = Oracle(pos, L)
    orc.build_precond()
    x = random_vec(6 * N, 4).astype(np.float32)
    g = st.precond_apply(_t(x)).cpu().numpy()
    assert rel_err(g, orc.precond_apply_jacobi(x, k)) < 1e-4
    b = random_vec(17 * N, 5).astype(np.float32)
    d = st.precond_apply(_t(b[:6 * N] - b[11 * N:])).cpu().numpy()
    xs = st.saddle_precond(_t(b)).cpu().numpy()
    ref = np.concatenate([b[:6 * N] - d, b[6 * N:11 * N], d])
    assert rel_err(xs, ref) < 1e-6

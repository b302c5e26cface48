"""Orthogonalisation kernels of GMRES and Lanczos at the edges of their forms.

Vectors of 17 N numbers: 2057 (three blocks, not a multiple of four), 131070 and 131087 (either side
of the line between the short and the long form, neither a multiple of four), 139264 (16-byte accesses).
GMRES's residual is an estimate from the Hessenberg matrix; it is the residual of the solution only if
the basis is orthonormal and the coefficients are those of the projections.  The solve stops at an
estimate of 1e-4 and the residual formed from its solution with FP32 products, whose rounding is of
the order of 1e-6, may be 10 % above that.  Once or twice projected, the solves take the same number of
iterations but for the one that rounding may shift.

Lanczos takes one coefficient of each projection only.  Its square roots with vectors of 131087 and 131120
(11 N), 131082 and 131088 numbers (6 N), just beyond the line and either a multiple of four or not, against
the same rule in 64 bits over the GPU's own products: equal but for the rounding of the products, or for one
step more where that shifts the stopping rule (a relative change of 1e-3).
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [121, 7710, 7711, 8192])
def test_residual_estimate(N):
    from fsd_amd.stokes import Stokes
    n = int(np.ceil(N ** (1 / 3)))
    L = 2.6 * n
    rng = np.random.default_rng(N)
    cell = np.stack(np.meshgrid(*[np.arange(n)] * 3, indexing="ij"), -1).reshape(-1, 3)[:N]
    pos = (cell + 0.5) * 2.6 - L / 2 + rng.uniform(-0.25, 0.25, (N, 3))
    p4 = torch.tensor(np.concatenate([pos, np.zeros((N, 1))], 1).astype(np.float32), device="cuda")
    b = torch.tensor(rng.standard_normal(17 * N).astype(np.float32), device="cuda")
    its = []
    for passes in (1, 2):
        st = Stokes(N, L, gmres_true_tol=1e-4, gram_schmidt_passes=passes)
        st.build_nlist(p4)
        st.build_precond(p4)
        x, info = st.saddle_solve(p4, b)
        r = b.double() - st.saddle_multiply(p4, x).double()
        assert info["converged"]
        assert (r.norm() / b.double().norm()).item() <= 1.1e-4
        its.append(info["iterations"])
    assert abs(its[0] - its[1]) <= 1 and its[0] > 8      # more than one group of eight vectors


@pytest.mark.parametrize("field,N", [("far", 11917), ("far", 11920), ("near", 21847), ("near", 21848)])
def test_long_lanczos(field, N):
    from fsd_amd.stokes import Stokes
    from oracle.oracle import lanczos_sqrt_adaptive
    n = int(np.ceil(N ** (1 / 3)))
    L = 2.6 * n
    rng = np.random.default_rng(N)
    cell = np.stack(np.meshgrid(*[np.arange(n)] * 3, indexing="ij"), -1).reshape(-1, 3)[:N]
    pos = (cell + 0.5) * 2.6 - L / 2 + rng.uniform(-0.25, 0.25, (N, 3))
    p4 = torch.tensor(np.concatenate([pos, np.zeros((N, 1))], 1).astype(np.float32), device="cuda")
    T, dt = 1.0, 1e-3
    st = Stokes(N, L, T=T, dt=dt)
    st.build_nlist(p4)
    m = 11 if field == "far" else 6
    psi = rng.standard_normal(m * N).astype(np.float32)
    noise = torch.tensor(psi, device="cuda")
    print("long Lanczos", field, N, flush=True)
    if field == "far":
        i = st.pse_info()
        st.set_noise(noise, torch.zeros(6 * i["Nx"] * i["Ny"] * i["Nz"], device="cuda"), None, None)
        y = st.brownian_farfield(p4)
        op = lambda v: st.mobility(p4, torch.tensor(v, dtype=torch.float32, device="cuda"), 1)  # noqa: E731
    else:
        st.set_noise(None, None, noise, None)
        y = st.brownian_nearfield(p4)
        op = lambda v: st.rfu(p4, torch.tensor(v, dtype=torch.float32, device="cuda"))  # noqa: E731
    ref, steps = lanczos_sqrt_adaptive(lambda v: op(v).double().cpu().numpy(), np.sqrt(2 * T / dt) * psi.astype(np.float64),
                                       2, 1e-3)
    assert steps > 2
    y = y.double().cpu().numpy()
    assert np.linalg.norm(y - ref) <= 1e-3 * np.linalg.norm(ref)


@pytest.mark.parametrize("N", [1001, 6000])
def test_two_passes_of_many_vectors(N):
    """two projections on more than 20 vectors, where N = 6000 (102000 numbers) goes from one form to the other
    on the way: the residual estimate as above, and up to 60 vectors take about 1.6 times as long as one
    projection, 34 and 21 us in the mean; where blocks go through all vectors twice, 43 us; 1.8 times is allowed"""
    from fsd_amd.stokes import Stokes
    n = int(np.ceil(N ** (1 / 3)))
    L = 2.6 * n
    rng = np.random.default_rng(N)
    cell = np.stack(np.meshgrid(*[np.arange(n)] * 3, indexing="ij"), -1).reshape(-1, 3)[:N]
    pos = (cell + 0.5) * 2.6 - L / 2 + rng.uniform(-0.25, 0.25, (N, 3))
    p4 = torch.tensor(np.concatenate([pos, np.zeros((N, 1))], 1).astype(np.float32), device="cuda")
    b = torch.tensor(rng.standard_normal(17 * N).astype(np.float32), device="cuda")
    us, its = [], []
    for passes in (1, 2):
        st = Stokes(N, L, gmres_true_tol=1e-5, gmres_restart=100, gram_schmidt_passes=passes, precond="ichol_jacobi",
                    jacobi_iters=1)
        st.build_nlist(p4)
        st.build_precond(p4)
        x, info = st.saddle_solve(p4, b)
        r = b.double() - st.saddle_multiply(p4, x).double()
        assert info["converged"] and info["restarts"] == 1
        assert (r.norm() / b.double().norm()).item() <= 1.1e-5
        its.append(info["iterations"])
        st = Stokes(N, L, gmres_tol=1e-12, gmres_maxiter=60, gmres_restart=60, gram_schmidt_passes=passes,
                    precond="ichol_jacobi", jacobi_iters=1)
        st.build_nlist(p4)
        st.build_precond(p4)
        st.saddle_solve(p4, b)
        st.profile(True, classes=["gmres_vec"])
        best = 1e30
        for _ in range(5):
            st.profile_reset()
            st.saddle_solve(p4, b)
            count, ms = st.profile_get("gmres_vec")
            best = min(best, 1e3 * ms / count)
        us.append(best)
    print("one and two passes", N, its, us)
    assert abs(its[0] - its[1]) <= 1 and its[0] > 20
    if N == 6000:
        assert us[1] < 1.8 * us[0]

"""Workloads that the performance of this framework is measured on.

``listed()`` names them, ``draw(rng)`` gives more of the same ranges, ``prepare``
makes what a program holds before the call (inputs on the GPU and the ``Stokes``
object with its tables, neighbour list and, where the call needs it, the
preconditioner), ``run`` makes the call, ``work`` says what the call cannot do
without and ``exact`` what it returns in 64 bits.

Sizes are those of the package's configurations and tests: suspensions of 343,
4096, 32768 and 262144 spheres at volume fractions 0.1 to 0.5, and the ensemble's
range of 200 to 2000.  A suspension is a random packing of ``n`` spheres, repeated
``rep`` times along each axis (``rep ** 3 n`` spheres in all) with every sphere then
displaced a little, so that no two parts of it are alike; ``lattice`` starts from the
jittered simple cubic lattice of the active suspension.  ``tilt`` deforms the
periodic box by ``tilt / rep``, which such a repeated packing fits without overlaps.
"""
import math

import numpy as np
import torch

from fsd_amd.stokes import ParticleState, Stokes
from fsd_amd.tables import load_resistance_table
from fsd_amd.workloads import jittered_lattice, random_forces, random_packing

GAP = 4e-3          # least gap of the packed spheres ...
JITTER = 7e-4       # ... and the displacement along each axis, which leaves at least GAP - 2 sqrt(3) JITTER


def listed():
    def case(name, kind, n, phi, rep=1, tilt=0, mode="ichol", lattice=False):
        return dict(name=name, kind=kind, n=n, phi=phi, rep=rep, tilt=tilt, mode=mode, lattice=lattice)
    return [
        # one far-field mobility product M F: the smallest suspension, where launches and latency count
        case("mobility-343", "mobility", 343, 0.20),
        # a sheared suspension in a deformed box, as an oscillatory or start-up protocol has it
        case("mobility-4072-tilted", "mobility", 509, 0.30, rep=2, tilt=1),
        # the benchmark's size and density
        case("mobility-32768", "mobility", 512, 0.45, rep=4),
        # the active suspension's size (grid 135^3, an odd length)
        case("mobility-262144", "mobility", 64 ** 3, 0.40, lattice=True),
        # one product of the whole saddle-point operator (far field and lubrication) for a dilute,
        # ragged suspension: what a caller's own Krylov solver calls
        case("saddle-13797", "saddle", 511, 0.15, rep=3, tilt=-1),
        # the lubrication operators of a stresslet output (R_FU, R_FE, R_SU, R_SE), dense
        case("lubrication-9261", "lubrication", 343, 0.50, rep=3),
        # one application of the saddle preconditioner: the reference's exact triangular solves, ...
        case("precond-exact-4096", "precond", 512, 0.30, rep=2),
        # ... IC(0) by Jacobi iterations at the size of an ensemble's replica, ...
        case("precond-jacobi-700", "precond", 700, 0.40, mode="ichol_jacobi"),
        # ... and the learned factor at the benchmark's size
        case("precond-learned-32768", "precond", 512, 0.45, rep=4, mode="learned"),
        # the random slip velocity and force of a Brownian step
        case("brownian-4096", "brownian", 512, 0.30, rep=2),
        # whole time steps, their saddle solve refined until the velocities are determined to 32 bits:
        # a replica of an ensemble, ...
        case("step-1000", "step", 1000, 0.25, mode="ichol_jacobi"),
        # ... and the benchmark's suspension with its preconditioner
        case("step-32768", "step", 512, 0.45, rep=4, mode="learned"),
    ]


def draw(rng):
    """a suspension of 200 to 180000 spheres and one of the calls above on it"""
    kind = rng.choice(["mobility", "mobility", "mobility", "saddle", "lubrication", "precond", "precond", "brownian",
                       "step"])
    most = {"mobility": 180000, "step": 4500}.get(kind, 33000)
    mode = rng.choice(["ichol", "ichol_jacobi", "learned"]) if kind in ("precond", "step") else "ichol"
    phi = round(rng.uniform(0.1, 0.5), 3)
    # the far field's grid grows with the volume: no larger than the largest listed case's
    target = math.exp(rng.uniform(math.log(200), math.log(min(most, 262144 / 0.4 * phi))))
    rep = max(1, math.ceil((target / 1000) ** (1 / 3)))
    n = max(200, int(target / rep ** 3))
    tilt = rng.randint(-(rep // 2), rep // 2) if rep > 1 else 0
    return dict(kind=kind, n=n, phi=phi, rep=rep, tilt=tilt, mode=mode, lattice=False)


def count(case):
    return case["n"] * case["rep"] ** 3


def box_of(case, L):
    return (L, L, L, case["tilt"] / case["rep"], 0.0, 0.0)


def suspension(case, seed):
    """(positions float32[N, 3], edge of the box)"""
    if case["lattice"]:
        return jittered_lattice(round(case["n"] ** (1 / 3)), case["phi"], seed=seed)
    base, L0 = random_packing(case["n"], case["phi"], seed=seed, min_gap=GAP)
    rep = case["rep"]
    L = L0 * rep
    shift = np.stack(np.meshgrid(*[np.arange(rep)] * 3, indexing="ij"), axis=-1).reshape(-1, 1, 3) * L0
    x = (base[None].astype(np.float64) + 0.5 * L0 + shift).reshape(-1, 3)
    x += np.random.default_rng(seed + 31).uniform(-JITTER, JITTER, size=x.shape)
    # into the box, whose top and bottom are displaced along x by the tilt
    y = np.mod(x[:, 1], L) - 0.5 * L
    turns = np.floor(x[:, 1] / L)
    lean = case["tilt"] / rep * y
    x0 = x[:, 0] - 0.5 * L - turns * case["tilt"] / rep * L - lean
    x0 = x0 - L * np.floor(x0 / L + 0.5) + lean
    z = np.mod(x[:, 2], L) - 0.5 * L
    return np.stack([x0, y, z], axis=1).astype(np.float32), float(L)


def inputs(case, seed):
    """the arrays a program hands over, on the GPU"""
    pos, L = suspension(case, seed)
    N = count(case)
    g = torch.Generator().manual_seed(seed)
    p4 = torch.zeros(N, 4)
    p4[:, :3] = torch.from_numpy(pos)
    s = dict(L=L, pos3=pos, pos=p4.reshape(-1).cuda())
    if case["kind"] == "mobility":            # forces, torques and stresslets
        s["x"] = torch.randn(11 * N, generator=g).cuda()
    elif case["kind"] == "lubrication":       # velocities
        s["x"] = torch.randn(6 * N, generator=g).cuda()
    elif case["kind"] in ("saddle", "precond"):
        s["x"] = torch.randn(17 * N, generator=g).cuda()
    elif case["kind"] == "step":
        s["x"] = torch.from_numpy(random_forces(N, seed=seed)).cuda()
    return s


def options(case):
    """the solver settings of the benchmark and of the ensemble for each preconditioner"""
    opt = dict(precond=case["mode"])
    if case["mode"] == "ichol_jacobi":
        opt.update(jacobi_iters=8)
    elif case["mode"] == "learned":
        opt.update(jacobi_iters=5, fallback_jacobi=8, learned_calibration=20)
    if case["kind"] == "step":
        opt.update(dt=1e-3, gmres_tol=1e-6, gmres_true_tol=2e-7, refine=True, gmres_restart=100, gmres_maxiter=4000,
                   gram_schmidt_passes=1, guess="extrapolate")
    elif case["kind"] == "brownian":
        opt.update(T=1.0, seed=7)
    return opt


def prepare(case, seed):
    s = inputs(case, seed)
    s["kind"] = case["kind"]
    s["stokes"] = st = Stokes(count(case), box_of(case, s["L"]), **options(case))
    if case["kind"] == "step":
        s["state"], s["step"] = ParticleState(s["pos3"]), 0
        return s
    st.build_nlist(s["pos"])
    if case["kind"] == "precond":
        st.build_precond(s["pos"])
    return s


def run(s):
    st, pos, x = s["stokes"], s["pos"], s.get("x")
    if s["kind"] == "mobility":
        return st.mobility(pos, x)
    if s["kind"] == "saddle":
        return st.saddle_multiply(pos, x)
    if s["kind"] == "lubrication":
        return dict(rfu=st.rfu(pos, x), rfe=st.rfe(pos, 1.0), rsu=st.rsu(pos, x), rse=st.rse(pos, 1.0))
    if s["kind"] == "precond":
        return st.saddle_precond(x)
    if s["kind"] == "brownian":
        return dict(slip=st.brownian_farfield(pos, 1), force=st.brownian_nearfield(pos, 1))
    st.integrateStepOne(s["step"], s["state"], force6=x, shear_rate=1.0)
    s["step"] += 1
    return dict(velocity=s["state"].velocity, pos=s["state"].pos)


# ------------------------------------------------------------------ work
def grid_points(case):
    """points of the far field's grid: the next length with no prime factor above 5 of at least
    3 L / pi + 1 along each axis"""
    L = (count(case) * 4 / 3 * math.pi / case["phi"]) ** (1 / 3)
    m = max(8, int(3 * L / math.pi) + 1)
    while True:
        q = m
        for f in (2, 3, 5):
            while q % f == 0:
                q //= f
        if q == 1:
            return m ** 3
        m += 1


def work(case):
    """Inputs and outputs once.  Operations of a mobility product: 6^3 nodes by 11 fields per sphere to the
    grid and back, two real transforms of the 11 fields, the Green's function, about 200 for each pair within
    the real-space cutoff 5.26; of a lubrication product 60 per pair within 4; of a preconditioner
    application the 6 x 6 blocks of the pairs within 2.1 both ways.  Iterative calls take as many products
    as their solve is known to need: about 10 for the Brownian terms, 150 for a refined step."""
    N, M = count(case), grid_points(case)
    density = 3 * case["phi"] / (4 * math.pi)
    pairs = lambda r: N * (4 / 3 * math.pi * r ** 3 * density)  # noqa: E731
    mobility = N * 2 * 216 * 22 + 2 * 11 * 2.5 * M * math.log2(M) + 60 * M + 200 * pairs(5.26)
    lubrication = 60 * pairs(4.0) + 72 * N
    contacts = N * 8 * case["phi"]
    precond = (72 * contacts + 72 * N) * 2
    kind = case["kind"]
    if kind == "mobility":
        return dict(bytes=N * (16 + 44 + 44), flops=mobility)
    if kind == "saddle":
        return dict(bytes=N * (16 + 68 + 68), flops=mobility + lubrication)
    if kind == "lubrication":
        return dict(bytes=N * (16 + 24 + 24 + 24 + 20 + 20), flops=5 * lubrication)
    if kind == "precond":
        return dict(bytes=N * (68 + 68) + 144 * (contacts / 2 + N), flops=precond)
    if kind == "brownian":
        return dict(bytes=N * (16 + 44 + 24), flops=10 * (200 * pairs(5.26) + lubrication) + mobility)
    return dict(bytes=N * (16 + 24 + 44 + 16), flops=150 * (mobility + lubrication + precond))


# ----------------------------------------------------------------- exact
# The same sums in 64 bits with torch alone.  The method's tables (the Ewald splitting's functions, the
# resistance functions) and the parameters of its grid are inputs of the method; which pairs lie within a
# cutoff is decided in 32 bits, in the order of operations that defines it.
def pairs_within(pos, L, tilt, r):
    """(i, j, p_i - p_j (minimum image) in 64 bits, its length in 32 bits) of the ordered pairs closer than r"""
    N = pos.shape[0]
    dev = pos.device
    frac = pos.double().clone()
    frac[:, 0] -= tilt * frac[:, 1]
    frac = frac / L + 0.5
    nc = int(L / (r * math.sqrt(1 + tilt * tilt) + 1e-3))
    found = []

    def keep(i, j):
        d = pos[i] - pos[j]
        f32 = lambda v: torch.tensor(v, dtype=torch.float32, device=dev)  # noqa: E731
        Lf, iL, xy = f32(L), f32(1.0) / f32(L), f32(tilt)
        nz = torch.round(d[:, 2] * iL)
        dz = d[:, 2] - Lf * nz
        ny = torch.round(d[:, 1] * iL)
        dx = d[:, 0] - (Lf * xy) * ny
        dy = d[:, 1] - Lf * ny
        nx = torch.round(dx * iL)
        dx = dx - Lf * nx
        d2 = dx * dx + dy * dy
        d2 = d2 + dz * dz
        near = (d2 < f32(r) * f32(r)) & (i != j)
        i, j, d2 = i[near], j[near], d2[near]
        e = pos[i].double() - pos[j].double()
        n = [v[near].double() for v in (nx, ny, nz)]
        edge = float(Lf)
        e[:, 2] -= edge * n[2]
        e[:, 1] -= edge * n[1]
        e[:, 0] -= edge * (float(xy) * n[1] + n[0])
        found.append((i, j, e, torch.sqrt(d2)))

    if nc < 3:
        every = torch.arange(N, device=dev)
        for a in range(0, N, 512):
            i = every[a:a + 512]
            keep(i.repeat_interleave(N), every.repeat(len(i)))
    else:
        c = torch.clamp((frac * nc).long(), 0, nc - 1)
        cell = (c[:, 0] * nc + c[:, 1]) * nc + c[:, 2]
        order = torch.argsort(cell, stable=True)
        filled = torch.bincount(cell, minlength=nc ** 3)
        start = torch.cumsum(filled, 0) - filled
        width = int(filled.max())
        ids = torch.full((nc ** 3, width), -1, device=dev)
        ids[cell[order], torch.arange(N, device=dev) - start[cell[order]]] = order
        at = torch.arange(nc ** 3, device=dev)
        ax = torch.stack([at // (nc * nc), at // nc % nc, at % nc])
        for o in range(27):
            b = (ax + torch.tensor([[o // 9 - 1], [o // 3 % 3 - 1], [o % 3 - 1]], device=dev)) % nc
            other = ids[(b[0] * nc + b[1]) * nc + b[2]]
            i = ids[:, :, None].expand(-1, -1, width).reshape(-1)
            j = other[:, None, :].expand(-1, width, -1).reshape(-1)
            ok = (i >= 0) & (j >= 0)
            keep(i[ok], j[ok])
    return [torch.cat(v) for v in zip(*found)]


def couplets(x, N):
    """forces [N, 3] and couplets [N, 3, 3] of the generalised force"""
    F, T, S = x[:6 * N].view(N, 6)[:, :3], x[:6 * N].view(N, 6)[:, 3:], x[6 * N:11 * N].view(N, 5)
    C = torch.zeros(N, 3, 3, dtype=x.dtype, device=x.device)
    for k, (a, b) in enumerate([(0, 0), (0, 1), (0, 2), (1, 2), (1, 1)]):
        C[:, a, b] = S[:, k]
        C[:, b, a] = S[:, k]
    C[:, 2, 2] = -(S[:, 0] + S[:, 4])
    for a, b, t in [(0, 1, 2), (1, 2, 0), (2, 0, 1)]:      # minus half the torque's antisymmetric part
        C[:, a, b] -= 0.5 * T[:, t]
        C[:, b, a] += 0.5 * T[:, t]
    return F, C


def wave_space(pos, F, C, L, tilt, pse, xi=0.5):
    """velocity [N, 3] and its gradient [N, 3, 3] from the grid"""
    n, P, N, dev = pse["Nx"], pse["P"], pos.shape[0], pos.device
    f32 = np.float32
    # each sphere's first node, as the method defines it in 32 bits
    p = pos.cpu().numpy()
    half = f32(0.5) * f32(L)
    lean = (f32(0) - f32(0) * f32(tilt)) * p[:, 2] + f32(tilt) * p[:, 1]
    fr = np.stack([(p[:, 0] + half) - lean, p[:, 1] + half, p[:, 2] + half], 1) / f32(L) * f32(n)
    first = fr.astype(np.int64)
    o = first - P // 2 + 1 - (P % 2) * ((fr - first.astype(f32)) < f32(0.5))
    o = torch.from_numpy(o).to(dev)
    h, edge, xy = float(pse["gridh_x"]), float(f32(L)), float(f32(tilt))
    t = torch.arange(P, device=dev)
    node = [h * (o[:, a, None] + t).double() - 0.5 * edge for a in range(3)]
    q = pos.double()
    dy, dz = node[1] - q[:, 1, None], node[2] - q[:, 2, None]
    dx = node[0][:, :, None] + xy * node[1][:, None, :] - q[:, 0, None, None]
    a = float(pse["expfac"])
    w = torch.exp(-a * (dx * dx + (dy * dy)[:, None, :]))[..., None] * torch.exp(-a * dz * dz)[:, None, None, :]
    w = (float(pse["prefac"]) * w).reshape(N, -1)
    m = [(o[:, k, None] + t) % n for k in range(3)]
    at = ((m[0][:, :, None, None] * n + m[1][:, None, :, None]) * n + m[2][:, None, None, :]).reshape(N, -1)
    src = torch.cat([F, C.reshape(N, 9)], 1)
    k1 = torch.arange(n, device=dev, dtype=torch.float64)
    k1 = torch.where(k1 < (n + 1) // 2, k1, k1 - n)
    two_pi = float(f32(2 * 3.1416926536))     # the reference's constant
    kx = (k1 / edge * two_pi)[:, None, None].expand(n, n, n)
    ky = ((k1[None, :, None] - xy * k1[:, None, None]) / edge * two_pi).expand(n, n, n)
    kz = (k1 / edge * two_pi)[None, None, :].expand(n, n, n)
    k = [kx, ky, kz]
    ksq = kx * kx + ky * ky + kz * kz
    ksq[0, 0, 0] = 1.0
    kk = torch.sqrt(ksq)
    G = 6 * 3.1415926536 * (1 + ksq / (4 * xi * xi)) * torch.exp(-(1 - float(pse["eta"])) * ksq / (4 * xi * xi)) / ksq
    G = G / n ** 3
    G[0, 0, 0] = 0.0
    j0 = torch.sin(kk) / kk
    j1 = 3 * (torch.sin(kk) - kk * torch.cos(kk)) / (ksq * kk)
    spec = []
    for c in range(12):
        grid = torch.zeros(n ** 3, dtype=torch.float64, device=dev)
        for s in range(0, N, 32768):
            grid.index_add_(0, at[s:s + 32768].reshape(-1), (w[s:s + 32768] * src[s:s + 32768, c, None]).reshape(-1))
        spec.append(torch.fft.fftn(grid.view(n, n, n)))
    f, cm = spec[:3], [spec[3 + 3 * r:6 + 3 * r] for r in range(3)]
    kf = (k[0] * f[0] + k[1] * f[1] + k[2] * f[2]) / ksq
    ck = [cm[r][0] * k[0] + cm[r][1] * k[1] + cm[r][2] * k[2] for r in range(3)]
    kck = (k[0] * ck[0] + k[1] * ck[1] + k[2] * ck[2]) / ksq
    # the field that moves a point force, and its smoothed forms (j0 for forces, j1 for couplets)
    v = [G * ((f[r] - k[r] * kf) * j0 - 1j * (ck[r] - k[r] * kck) * j1) for r in range(3)]
    del spec, f, cm, ck, kck, kf

    def at_spheres(field):
        real = torch.fft.ifftn(field).real.reshape(-1) * n ** 3
        out = torch.empty(N, dtype=torch.float64, device=dev)
        for s in range(0, N, 32768):
            out[s:s + 32768] = (real[at[s:s + 32768]] * w[s:s + 32768]).sum(1)
        return out * float(pse["quadW"])

    u = torch.stack([at_spheres(v[r] * j0) for r in range(3)], 1)
    D = torch.stack([torch.stack([at_spheres(1j * v[r] * k[c] * j1) for c in range(3)], 1) for r in range(3)], 1)
    return u, D


def real_space(pos, F, C, L, tilt, pse, table):
    """velocity and its gradient from the pairs within the cutoff, and each sphere's own part"""
    i, j, e, d32 = pairs_within(pos, L, tilt, float(pse["rcut"]))
    dr, rc, n = float(np.float32(0.001)), float(pse["rcut"]), pse["ewald_n"]
    u = float(pse["self_x"]) * F
    D = float(pse["self_y"]) * (C - 4 * C.transpose(1, 2))
    for s in range(0, len(i), 1 << 21):
        a, b, d = i[s:s + (1 << 21)], j[s:s + (1 << 21)], e[s:s + (1 << 21)]
        r = torch.sqrt((d * d).sum(1))
        row = torch.clamp(torch.floor((r - dr) * (n / (rc - dr))).long(), 0, n - 1)
        f = table[row] + (table[row + 1] - table[row]) * (r / dr - row - 1)[:, None]
        f1, f2, g1, g2, h1, h2, h3 = [f[:, k, None] for k in range(7)]
        g1, g2 = -g1, -g2
        R = d / r[:, None]
        Fj, Cj = F[b], C[b]
        rF = (R * Fj).sum(1, keepdim=True)
        Cr = torch.einsum("nab,nb->na", Cj, R)
        rC = torch.einsum("nba,nb->na", Cj, R)
        rCr = (R * Cr).sum(1, keepdim=True)
        u.index_add_(0, a, f1 * Fj + (f2 - f1) * rF * R + g1 * (Cr - rCr * R) + g2 * (rC - 4 * rCr * R))
        out = lambda x, y: x[:, :, None] * y[:, None, :]  # noqa: E731
        one = torch.eye(3, dtype=pos.double().dtype, device=pos.device)[None]
        RR, w = out(R, R), lambda v: v[:, :, None]        # noqa: E731
        D.index_add_(0, a, -w(g1) * (out(R, Fj) - w(rF) * RR) - w(g2) * (one * w(rF) + out(Fj, R) - 4 * w(rF) * RR)
                     + w(h1) * (Cj - 4 * Cj.transpose(1, 2)) + w(h2) * (out(R, Cr) - w(rCr) * RR)
                     + w(h3) * (one * w(rCr) + out(Cr, R) + out(R, rC) + out(rC, R) - 6 * w(rCr) * RR
                                - Cj.transpose(1, 2)))
    return u, D


def mobility64(pos, x, case, L):
    """generalised velocity 11N of the generalised force 11N"""
    N, tilt = pos.shape[0], case["tilt"] / case["rep"]
    st = Stokes(N, box_of(case, L))
    pse = st.pse_info()
    table = torch.from_numpy(st.get_ewald_table()).double().cuda().view(-1, 8)
    del st
    F, C = couplets(x.double(), N)
    u, D = real_space(pos, F, C, L, tilt, pse, table)
    uw, Dw = wave_space(pos, F, C, L, tilt, pse)
    u, D = u + uw, D + Dw.transpose(1, 2)
    W = 0.5 * torch.stack([D[:, 1, 2] - D[:, 2, 1], D[:, 2, 0] - D[:, 0, 2], D[:, 0, 1] - D[:, 1, 0]], 1)
    E = 0.5 * (D + D.transpose(1, 2))
    S = torch.stack([2 * E[:, 0, 0] + E[:, 1, 1], 2 * E[:, 0, 1], 2 * E[:, 0, 2], 2 * E[:, 1, 2],
                     2 * E[:, 1, 1] + E[:, 0, 0]], 1)
    return torch.cat([torch.cat([u, W], 1).reshape(-1), S.reshape(-1)])


def resistances(pos, L, tilt):
    """(i, j, unit vector from i to j, the 22 resistance functions) of the pairs within 4"""
    i, j, e, d32 = pairs_within(pos, L, tilt, 4.0)
    dist, vals = [torch.from_numpy(np.asarray(v, dtype=np.float32)).double().cuda() for v in load_resistance_table()]
    vals = vals.view(1000, 22)
    r = torch.sqrt((e * e).sum(1))
    close = d32.double() <= 2.001
    step = float(np.float32(0.004305))
    row = torch.clamp((torch.log10(torch.clamp(r - 2, min=1e-9) / 1e-4) / step).long(), 0, 999)
    up = torch.clamp(row + 1, max=999)
    fac = torch.where(row < 999, (r - dist[row]) / (dist[up] - dist[row] + (row == 999)), 0.0)
    v = vals[row] + (vals[up] - vals[row]) * fac[:, None]
    return i, j, -e / r[:, None], torch.where(close[:, None], vals[232][None], v)


def turn(r, v):
    """eps . r . v"""
    return torch.linalg.cross(v, r)


def rfu64(pos, U, L, tilt, res=None):
    N = pos.shape[0]
    i, j, r, v = res or resistances(pos, L, tilt)
    f = [v[:, k, None] for k in range(10)]
    U = U.double().view(N, 6)
    dot = lambda a, b: (a * b).sum(1, keepdim=True)  # noqa: E731
    ui, wi, uj, wj = U[i, :3], U[i, 3:], U[j, :3], U[j, 3:]
    force = ((f[0] - f[2]) * dot(r, ui) * r + f[2] * ui - f[4] * turn(r, wi)
             + (f[1] - f[3]) * dot(r, uj) * r + f[3] * uj + f[5] * turn(r, wj))
    torque = (f[4] * turn(r, ui) + (f[6] - f[8]) * dot(r, wi) * r + f[8] * wi
              + f[5] * turn(r, uj) + (f[7] - f[9]) * dot(r, wj) * r + f[9] * wj)
    out = torch.zeros(N, 6, dtype=torch.float64, device=pos.device)
    return out.index_add_(0, i, torch.cat([force, torque], 1)).reshape(-1)


def lubrication64(pos, U, L, tilt, rate):
    N = pos.shape[0]
    i, j, r, v = res = resistances(pos, L, tilt)
    XG11, XG12, YG11, YG12, YH11, YH12, XM11, XM12, YM11, YM12, ZM11, ZM12 = [v[:, k, None] for k in range(10, 22)]
    E = torch.zeros(3, 3, dtype=torch.float64, device=pos.device)
    E[0, 1] = E[1, 0] = 0.5 * rate
    dot = lambda a, b: (a * b).sum(1, keepdim=True)  # noqa: E731
    Er = r @ E
    rEr, eEr = dot(r, Er), turn(r, Er)
    zero = lambda k: torch.zeros(N, k, dtype=torch.float64, device=pos.device)  # noqa: E731
    # the second sphere of a pair sees XG21 = -XG12, YG21 = -YG12, YH21 = YH12
    force = (-(XG11 - 2 * YG11) + (XG12 - 2 * YG12)) * rEr * r + 2 * (YG12 - YG11) * Er
    rfe = zero(6).index_add_(0, i, torch.cat([force, 2 * (YH11 + YH12) * eEr], 1))
    U = U.double().view(N, 6)
    sym = [(0, 0), (0, 1), (0, 2), (1, 2), (1, 1)]
    rsu, rse = [], []
    for a, b in sym:
        third = 1 / 3 if a == b else 0.0
        A, B = slice(a, a + 1), slice(b, b + 1)
        rr = r[:, A] * r[:, B]
        s = 0.0
        for u, w, XG, YG, YH in ((U[i, :3], U[i, 3:], XG11, YG11, YH11), (U[j, :3], U[j, 3:], XG12, YG12, YH12)):
            ru, ew = dot(r, u), turn(r, w)
            s = s + XG * (rr - third) * ru + YG * (u[:, A] * r[:, B] + r[:, A] * u[:, B] - 2 * rr * ru)
            s = s + YH * (r[:, A] * ew[:, B] + ew[:, A] * r[:, B])
        rsu.append(s)
        cross = r[:, A] * Er[:, B] + r[:, B] * Er[:, A]
        rse.append(1.5 * (XM11 + XM12) * (rr - third) * rEr + (YM11 + YM12) * (cross - 2 * rEr * rr)
                   + 0.5 * (ZM11 + ZM12) * (2 * E[a, b] + (float(a == b) + rr) * rEr - 2 * cross))
    return dict(rfu=rfu64(pos, U, L, tilt, res), rfe=rfe.reshape(-1),
                rsu=-zero(5).index_add_(0, i, torch.cat(rsu, 1)).reshape(-1),
                rse=zero(5).index_add_(0, i, torch.cat(rse, 1)).reshape(-1))


def exact(case, seed):
    """Products and operators.  None for a preconditioner (its value is the result of a factorisation that
    drops entries, in an order found on the host), for the Brownian terms (square roots up to a tolerance) and
    for a step (an iterate that stops at a residual)."""
    if case["kind"] not in ("mobility", "saddle", "lubrication"):
        return None
    s = inputs(case, seed)
    pos, N, tilt = s["pos"].view(-1, 4)[:, :3].contiguous(), count(case), case["tilt"] / case["rep"]
    if case["kind"] == "mobility":
        return mobility64(pos, s["x"], case, s["L"])
    if case["kind"] == "lubrication":
        return lubrication64(pos, s["x"], s["L"], tilt, 1.0)
    x = s["x"].double()
    y = mobility64(pos, x[:11 * N], case, s["L"])
    y[:6 * N] += x[11 * N:]
    return torch.cat([y, x[:6 * N] - rfu64(pos, x[11 * N:], s["L"], tilt)])

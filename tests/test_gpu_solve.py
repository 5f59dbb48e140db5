"""cms2d_solve (drop-in for the reference's solve) on a general cell list:
Cartesian lists with land cells (nmaxfaces 4), two-level telescoping lists
(nmaxfaces 6) and the scalar-transport system the salinity/heat callers build
(salinity.F90:510,599, heat.f90:480,559) from the flow's face fluxes."""
import ctypes as C

import numpy as np
import pytest

from cell_list import cart_cell_list, dense_system, tel_cell_list
from cms2d_amd import _lib, cases
from cms2d_amd.flow import FlowStep, solve, solve_adjoint
from pyoracle import D, I, Oracle, lib as olib


def make_system(seed, nx=24, ny=18, land=0.15):
    rng = np.random.default_rng(seed)
    act = rng.random((ny, nx)) > land
    n, nd, c2c = cart_cell_list(act)
    acoef = np.zeros((nd, 4))
    acoef[:n] = rng.uniform(0.2, 2.0, (n, 4))
    sp = np.zeros(nd)
    sp[:n] = -rng.uniform(0.05, 0.5, n)
    ss = np.zeros(nd)
    ss[:n] = rng.normal(size=n)
    phi = np.zeros(nd)
    phi[:n] = rng.normal(scale=0.1, size=n)
    phi[n:] = rng.normal(size=nd - n)
    iwet = np.ones(nd, dtype=np.int32)
    return n, nd, c2c, acoef, sp, ss, phi, iwet


@pytest.mark.gpu
@pytest.mark.parametrize("seed,relax", [(0, 1.0), (1, 0.8), (2, 1.0)])
def test_solve_matches_dense_and_oracle(gpu_available, seed, relax):
    n, nd, c2c, acoef, sp, ss, phi, iwet = make_system(seed)
    print(f"solve seed {seed} relax {relax} n {n}", flush=True)
    A, b = dense_system(n, acoef, c2c, sp, ss, phi, relax)
    x = np.linalg.solve(A, b + 1e-15 * 0)
    ss_g, phi_g = ss.copy(), phi.copy()
    res_g, rmom_g, it_g = solve(acoef, c2c, iwet, ss_g, sp, phi_g, relax, ncells=n)
    ss_o, phi_o, res_o = ss.copy(), phi.copy(), np.zeros(nd)
    rm = C.c_double()
    olib().cms_oracle_solve(n, nd, 4, acoef.ctypes.data_as(D), c2c.ctypes.data_as(I),
                            iwet.ctypes.data_as(I), ss_o.ctypes.data_as(D), sp.ctypes.data_as(D),
                            res_o.ctypes.data_as(D), phi_o.ctypes.data_as(D), relax, 1e-10, 1e-12,
                            4000, C.byref(rm))
    scale = np.abs(x).max()
    assert np.abs(phi_g[:n] - x).max() <= 1e-8 * scale
    assert np.abs(phi_o[:n] - x).max() <= 1e-8 * scale
    assert np.array_equal(phi_g[n:], phi[n:])                 # ghosts untouched
    assert np.abs(rmom_g - rm.value) <= 1e-12 * max(rm.value, 1e-30)
    assert np.abs(res_g[:n] - res_o[:n]).max() <= 1e-12 * np.abs(res_o).max()
    assert np.abs(ss_g[:n] - ss_o[:n]).max() <= 1e-13 * np.abs(ss_o).max()
    assert it_g > 0


def oracle_solve(n, nd, acoef, c2c, iwet, ss, sp, phi, relax):
    ss_o, phi_o, res_o = ss.copy(), phi.copy(), np.zeros(nd)
    rm = C.c_double()
    it = olib().cms_oracle_solve(n, nd, acoef.shape[1], acoef.ctypes.data_as(D),
                                 c2c.ctypes.data_as(I), iwet.ctypes.data_as(I),
                                 ss_o.ctypes.data_as(D), sp.ctypes.data_as(D),
                                 res_o.ctypes.data_as(D), phi_o.ctypes.data_as(D), relax, 1e-10,
                                 1e-12, 4000, C.byref(rm))
    assert it > 0
    return ss_o, phi_o, res_o, rm.value


def check_against(n, nd, c2c, acoef, sp, ss, phi, iwet, relax):
    A, b = dense_system(n, acoef, c2c, sp, ss, phi, relax)
    x = np.linalg.solve(A, b)
    ss_g, phi_g = ss.copy(), phi.copy()
    res_g, rmom_g, it_g = solve(acoef, c2c, iwet, ss_g, sp, phi_g, relax, ncells=n)
    ss_o, phi_o, res_o, rm = oracle_solve(n, nd, acoef, c2c, iwet, ss, sp, phi, relax)
    scale = np.abs(x).max()
    assert np.abs(phi_g[:n] - x).max() <= 1e-8 * scale
    assert np.abs(phi_o[:n] - x).max() <= 1e-8 * scale
    assert np.array_equal(phi_g[n:], phi[n:])
    assert np.abs(rmom_g - rm) <= 1e-12 * max(rm, 1e-30)
    assert np.abs(res_g[:n] - res_o[:n]).max() <= 1e-12 * np.abs(res_o).max()
    assert np.abs(ss_g[:n] - ss_o[:n]).max() <= 1e-13 * np.abs(ss_o).max()
    assert it_g > 0


@pytest.mark.gpu
@pytest.mark.parametrize("seed", [0, 1])
def test_solve_telescoping_cell_list(gpu_available, seed):
    """nmaxfaces = 6; a coarse cell in the inner corner of the refined region
    has two fine neighbours on two sides."""
    rng = np.random.default_rng(seed)
    refined = np.zeros((30, 40), bool)
    refined[6:20, 0:14] = True
    refined[18:26, 12:22] = True
    n, nd, c2c, level, _ = tel_cell_list(refined)
    assert (c2c[:n] >= 0).sum(1).max() == 6
    print(f"telescoping solve seed {seed}: {n} cells, {nd - n} ghosts", flush=True)
    acoef = np.where(c2c >= 0, rng.uniform(0.2, 2.0, c2c.shape), 0.0)
    acoef[n:] = 0.0
    sp = np.zeros(nd)
    sp[:n] = -rng.uniform(0.05, 0.5, n)
    ss = np.zeros(nd)
    ss[:n] = rng.normal(size=n)
    phi = rng.normal(scale=0.1, size=nd)
    check_against(n, nd, c2c, acoef, sp, ss, phi, np.ones(nd, dtype=np.int32), 1.0)


@pytest.mark.gpu
def test_solve_scalar_transport_system(gpu_available):
    """Implicit advection-diffusion of a scalar (salinity) over one flow step:
    a_k = K hk ds/dn + max(-F_k, 0) (upwind, Patankar's form), ap = sum a -
    sp with the storage sp = -A h/dt, ss = A h1 c1/dt, the boundary value on
    the ghost cells; F_k, hk and h from 20 steps of the 80x48 basin."""
    c = cases.basin(nx=80, ny=48, dx=10.0, seed=4, dt=60.0)
    o = Oracle(c, serial=0)
    h1 = o.get("h").copy()
    for _ in range(20):
        assert o.step(1)[0] == 0
    flux, hk, h = o.get_face("flux"), o.get_face("hk"), o.get("h")
    n, nd, c2c = cart_cell_list(np.ones((c.ny, c.nx), bool))
    area, kdiff = c.dx * c.dy, 1.0
    acoef = np.zeros((nd, 4))
    acoef[:n] = kdiff * hk * (c.dx / c.dx) + np.maximum(-flux, 0.0)   # ds/dn = 1 on a uniform grid
    rng = np.random.default_rng(5)
    c1 = 30.0 + 5.0 * rng.random(n)
    sp = np.zeros(nd)
    sp[:n] = -area * h / c.dt
    ss = np.zeros(nd)
    ss[:n] = area * h1 * c1 / c.dt
    phi = np.full(nd, 35.0)                 # ocean salinity on the ghost cells
    phi[:n] = c1
    print(f"transport system {n} cells", flush=True)
    check_against(n, nd, c2c, acoef, sp, ss, phi, np.ones(nd, dtype=np.int32), 1.0)


@pytest.mark.gpu
def test_jacobi_iterations_within_five_times_block_lu():
    """The GPU solve's Jacobi-BiCGStab on a 6-face telescoping list with a
    pp-like system (storage 0.3 % of the face coefficients) needs fewer than
    5x the iterations of BiCGStab preconditioned by exact (dense LU) solves of
    blocks of 64 consecutive cells, the block-Jacobi bound ILU(0) in those
    blocks approaches."""
    import scipy.sparse as sps
    import scipy.sparse.linalg as sla

    from cell_list import dense_system, tel_cell_list
    rng = np.random.default_rng(1)
    refined = np.zeros((40, 60), dtype=bool)
    refined[10:30, 20:40] = True
    n, nd, c2c, _, _ = tel_cell_list(refined)
    nf = c2c.shape[1]
    acoef = np.where(c2c >= 0, rng.uniform(0.5, 2.0, (nd, nf)), 0.0)
    acoef[n:] = 0.0
    sp = np.zeros(nd)
    sp[:n] = -0.003 * acoef[:n].sum(axis=1)
    ss = np.zeros(nd)
    ss[:n] = rng.normal(size=n)
    phi = np.zeros(nd)
    A, b = dense_system(n, acoef, c2c, sp, ss, phi, 1.0)
    blocks = [(s, min(n, s + 64)) for s in range(0, n, 64)]
    inv = [np.linalg.inv(A[s:e, s:e]) for s, e in blocks]

    def block_lu(r):
        z = np.empty_like(r)
        for (s, e), m in zip(blocks, inv):
            z[s:e] = m @ r[s:e]
        return z

    it = [0]
    sla.bicgstab(sps.csr_matrix(A), b, M=sla.LinearOperator((n, n), matvec=block_lu), rtol=1e-10, atol=0,
                 maxiter=5000, callback=lambda xk: it.__setitem__(0, it[0] + 1))
    _, _, it_g = solve(acoef, c2c, np.ones(nd, dtype=np.int32), ss.copy(), sp, phi.copy(), 1.0, ncells=n)
    print("GPU Jacobi-BiCGStab", it_g, "block dense-LU BiCGStab", it[0], flush=True)
    assert it_g < 5 * it[0]


def _flow_fields(c, steps, **kw):
    g = FlowStep(c, **kw)
    kry = [g.step(1)["kry"] for _ in range(steps)]
    out = [g.get(n) for n in ("eta", "u", "v", "p")]
    g.close()
    return kry, out


def _list_solves(faces):
    if faces == 4:
        n, nd, c2c, acoef, sp, ss, phi, iwet = make_system(7, nx=61, ny=43)
    else:
        refined = np.zeros((30, 40), bool)
        refined[6:20, 0:14] = True
        n, nd, c2c, _, _ = tel_cell_list(refined)
        rng = np.random.default_rng(8)
        acoef = np.where(c2c >= 0, rng.uniform(0.2, 2.0, c2c.shape), 0.0)
        acoef[n:] = 0.0
        sp, ss, phi, iwet = np.zeros(nd), np.zeros(nd), rng.normal(size=nd), np.ones(nd, dtype=np.int32)
        sp[:n], ss[:n] = -rng.uniform(0.05, 0.5, n), rng.normal(size=n)
    p = phi.copy()
    res, rmom, it = solve(acoef, c2c, iwet, ss, sp, p, 0.8, ncells=n)
    *grads, itg = solve_adjoint(acoef, c2c, sp, phi, p, 0.8, np.random.default_rng(9).normal(size=n), ncells=n)
    return [it, itg], [p, ss, res, *grads]


FUSED_FORMS = {
    "fp64": lambda: _flow_fields(cases.tidal(nx=70, ny=45, dx=20.0, seed=2), 6),
    "fp32": lambda: _flow_fields(cases.tidal(nx=70, ny=45, dx=20.0, seed=2), 6, precision=_lib.PREC_FP32_REFINE),
    "jacobi": lambda: _flow_fields(cases.basin(nx=40, ny=20, dx=10.0, seed=0), 6, precond=_lib.PRECOND_JACOBI),
    "strip": lambda: _flow_fields(cases.basin(nx=300, ny=5, dx=10.0, seed=0), 4, precond=_lib.PRECOND_JACOBI),
    "list4": lambda: _list_solves(4),
    "list6": lambda: _list_solves(6),
}


@pytest.mark.gpu
@pytest.mark.parametrize("form", list(FUSED_FORMS))
def test_three_launch_iteration_equals_five_sweeps(gpu_available, monkeypatch, form):
    """The Jacobi iteration in three launches (small systems) and in five
    (larger ones, here by CMS2D_FUSED_CELLS=0) form the same values in the same
    order: bitwise the same results and iteration counts for every solve that
    takes it -- u/v of the FP64 and FP32 forms, pp without a multigrid, cell
    lists of four and six faces and their reverse (the transposed u/v solves:
    test_gpu_step_adjoint.py)."""
    runs = []
    for cells in ("65536", "0"):
        monkeypatch.setenv("CMS2D_FUSED_CELLS", cells)
        print(f"fused up to {cells} cells, {form}", flush=True)
        runs.append(FUSED_FORMS[form]())
    assert runs[0][0] == runs[1][0]
    assert any(np.abs(a).max() > 0 for a in runs[0][1])
    for a, b in zip(runs[0][1], runs[1][1]):
        assert np.array_equal(a, b)

"""The default schedule (fused = 0) runs the reference's kernel sequence in fewer passes: against the kernels
called one by one (include/esdg.h), every array that both leave behind, bit for bit."""
import os

import numpy as np
import pytest

from esdgsem_mpiocca_amd import Case, RunParams
from esdgsem_mpiocca_amd import setup_api as S

pytestmark = pytest.mark.gpu

ISM_MESH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "meshes", "CircleInCircle.mesh")
RK_A, RK_C = (0.0, -5.0 / 9.0, -153.0 / 128.0), (1.0 / 3.0, 15.0 / 16.0, 8.0 / 15.0)   # low-storage RK3


@pytest.fixture(scope="module")
def dev():
    import esdgsem_mpiocca_amd as E
    return E.device()


def make(mesh, N):
    """(case, run parameters) of a mesh and its boundary: walls, inner/outer, ocean, periodic, or a general
    quad mesh with reversed faces."""
    if mesh == "ocean":
        return Case.ocean_uplift(N=N, nel=5), dict(bc_kind=2, h_zero=4000.0)
    if mesh == "periodic":
        return Case.gaussian_bump(N=N, nel=5), {}
    if mesh == "reversed":
        return Case.from_ism(ISM_MESH, N=N, case_kind=S.CASE_GAUSSIAN_BUMP, amp=0.05), {}
    return Case.dam_break(N=N, nel=5, noise=1e-3, seed=N), dict(bc_kind=1) if mesh == "inner" else {}


def by_kernels(ctx, case, rp, dts):
    a, E, F, ngl = case.arrays, case.Nelem, case.Nfaces, case.ngl
    nn, fn = E * ngl * ngl, F * ngl
    d = {k: ctx.array(v) for k, v in a.items()}
    met = (d["Jac"], d["yXi"], d["yEta"], d["xXi"], d["xEta"])
    conn = (d["ElemEdgeMasterSlave"], d["ElemEdgeOrientation"], d["ElemToEdge"])
    q, Qt, g = ctx.array(a["q"]), ctx.empty(nn * 3), ctx.array(np.zeros(nn * 3))
    qL, qR, SP, bL, bR = (ctx.empty(fn * k) for k in (3, 3, 3, 1, 1))
    zero = ctx.array(np.zeros(fn))
    gX, gY, SGX, SGY, XL, XR, YL, YR, SPV = (ctx.empty(n * 2) for n in [nn, nn] + [fn] * 7)
    V, VP, VL, VR = (ctx.empty(n) for n in (E, E, F, F))
    ctx.collect_edge_data_bottom(F, d["EdgeData"], d["b"], bL, bR)
    for dt in dts:
        for A, C in zip(RK_A, RK_C):
            ctx.collect_edge_data(F, d["EdgeData"], q, d["x"], d["y"], d["nx"], d["ny"], bL, bR, qL, qR, 0.0)
            ctx.volume_kernel(E, *met, q, d["D"], d["Bx"], d["By"], Qt)
            ctx.calc_num_fluxes(F, d["EdgeData"], d["EdgeReversed"], d["nx"], d["ny"], d["scal"], qL, qR, bL, bR, SP)
            ctx.surface_kernel(E, d["Jac"], *conn, SP, zero, zero, Qt)
            if rp.artificial_viscosity:
                ctx.shock_capturing(E, q, d["b"], d["VdmInv"], d["EleSizes"], V, VP)
                ctx.calc_num_fluxes_gradient(F, d["EdgeData"], d["nx"], d["ny"], d["scal"], qL, qR, SGX, SGY)
                ctx.calc_gradient(E, *met, q, d["b"], d["Dhat"], gX, gY)
                ctx.surface_kernel_gradient(E, d["Jac"], *conn, SGX, SGY, gX, gY)
                ctx.scale_gradient(E, q, gX, gY)
                ctx.collect_edge_data_gradient(F, d["EdgeData"], gX, gY, V, VL, VR, XL, XR, YL, YR)
                ctx.volume_kernel_viscose(E, *met, gX, gY, d["Dstrong"], V, Qt)
                ctx.calc_num_fluxes_viscose(F, d["EdgeData"], d["nx"], d["ny"], d["scal"], VL, VR, XL, XR, YL, YR, SPV)
                ctx.surface_kernel_visc(E, d["Jac"], *conn, SPV, Qt)
            ctx.calc_rk(E, Qt, A, 0.0, g)
            ctx.update_kernel_ls(E, C, dt, g, q)
            if rp.positivity:
                ctx.pos_pres(E, d["EleSizes"], d["w_GL"], d["Jac"], q)
    out = dict(q=q, Qt=Qt, gRK=g, qL=qL, qR=qR, SurfaceParts=SP)
    if rp.artificial_viscosity:
        out.update(qGradientX=gX, qGradientY=gY, ViscPara=V, ViscForPlot=VP)
    return {k: v.download().ravel() for k, v in out.items()}


def check(dev, case, rp, av):
    ctx = dev.Context(dev.make_params(case, rp))
    try:
        s = dev.Solver(ctx, case, rp, fused=0)
        dts = []
        for _ in range(2):
            assert s.run(1)[0] == 1
            dts.append(s.last_dt())
        ref = by_kernels(ctx, case, rp, dts)
        assert np.isfinite(ref["q"]).all()
        for name, v in ref.items():
            assert np.array_equal(s.view(name, v.size).download(), v), name
        if av:
            assert (ref["ViscPara"] > 0).any()
        s.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("av", [0, 1])
@pytest.mark.parametrize("N", range(1, 10))
def test_degrees(dev, N, av):
    if av and N == 1:
        pytest.skip("the sensor's two top shells need modes below them")
    case, kw = make("walls", N)
    check(dev, case, RunParams(num_flux=3, rk_order=3, artificial_viscosity=av, eps0=0.005, sigma_min=-4.5,
                               sigma_max=-2.5, DFL=0.05, **kw), av)


@pytest.mark.parametrize("flux", [0, 1, 3, 4, 5])
@pytest.mark.parametrize("mesh", ["walls", "inner", "ocean", "periodic", "reversed"])
def test_boundaries_and_fluxes(dev, mesh, flux):
    case, kw = make(mesh, 4)
    check(dev, case, RunParams(num_flux=flux, rk_order=3, **kw), 0)


@pytest.mark.parametrize("N", [4, 6])
def test_reversed_faces_with_viscosity(dev, N):
    case, kw = make("reversed", N)
    check(dev, case, RunParams(num_flux=3, rk_order=3, artificial_viscosity=1, eps0=0.005, sigma_min=-12.0,
                               sigma_max=-10.0, DFL=0.05, **kw), 1)


@pytest.mark.parametrize("av", [0, 1])
@pytest.mark.parametrize("N", [2, 5, 7])
def test_limiter(dev, N, av):
    case = Case.flood(N=N, nel=6, seed=2)
    check(dev, case, RunParams(num_flux=3, rk_order=3, positivity=1, pos_pres_tol=1e-3, CFL=0.1, eps0=0.005,
                               artificial_viscosity=av, sigma_min=-4.5, sigma_max=-2.5, DFL=0.05), av)

"""GPU parity of the whole time loop (deviceclass::DGtimeloop) against the oracle.

Acceptance bar: relative L2 <= 1e-12 after a fixed number of steps; lake at rest
keeps |u|, |v| <= 1e-13.
"""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

from esdgsem_mpiocca_amd import Case, RunParams, total_entropy, total_mass
from esdgsem_mpiocca_amd import setup_api as S
from helpers import rel_l2
from oracle import binding as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import esdgsem_mpiocca_amd as E
    return E.device()


SCHEDULES = [0, 1, 2]
SCHEDULE_IDS = ["reference_sequence", "fused", "single_kernel"]


def run_gpu(dev, case, rp, steps, fused=0):
    ctx = dev.Context(dev.make_params(case, rp))
    try:
        s = dev.Solver(ctx, case, rp, fused=fused)
        n, t = s.run(steps)
        q = s.get_q()
        s.close()
    finally:
        ctx.close()
    return q, n, t


def fields_rel_l2(case, a, b):
    A = a.reshape(case.Nelem, 3, -1)
    B = b.reshape(case.Nelem, 3, -1)
    return [rel_l2(A[:, v], B[:, v]) if np.linalg.norm(B[:, v]) > 0 else np.abs(A[:, v]).max()
            for v in range(3)]


@pytest.mark.parametrize("fused", SCHEDULES, ids=SCHEDULE_IDS)
def test_c0_bump_200_steps(dev, fused):
    """Periodic Cartesian 16x16, N=4, EC volume + ES surface, LSRK4, CFL 0.5, 200 steps."""
    case = Case.gaussian_bump(N=4, nel=16)
    rp = RunParams(num_flux=0)
    qo, no, to, _ = O.timeloop(case, rp, 200)
    qg, ng, tg = run_gpu(dev, case, rp, 200, fused=fused)
    assert ng == no == 200
    assert abs(tg - to) <= 1e-14 * to
    h, hu, hv = fields_rel_l2(case, qg, qo)
    assert h <= 1e-12 and hu <= 1e-12 and hv <= 1e-12, (h, hu, hv)


@pytest.mark.parametrize("fused", SCHEDULES, ids=SCHEDULE_IDS)
def test_c0_lake_at_rest(dev, fused):
    case = Case.gaussian_bump(N=4, nel=16, lake_at_rest=True)
    rp = RunParams(num_flux=0)
    qg, ng, _ = run_gpu(dev, case, rp, 200, fused=fused)
    Q = qg.reshape(case.Nelem, 3, -1)
    assert np.abs(Q[:, 1]).max() <= 1e-13 and np.abs(Q[:, 2]).max() <= 1e-13
    eta = Q[:, 0] + case["b"].reshape(case.Nelem, -1)
    assert np.abs(eta - 1.0).max() <= 1e-13
    assert abs(total_mass(case, qg) - total_mass(case, case["q"])) <= 1e-13


@pytest.mark.parametrize("fused", [0, 1], ids=SCHEDULE_IDS[:2])
def test_dam_break_curved_av(dev, fused):
    """Curved 12x12 N=7 dam break with modal sensor + artificial viscosity, rotated ES flux."""
    case = Case.dam_break(N=7, nel=12, noise=1e-3, seed=0)
    rp = RunParams(num_flux=3, artificial_viscosity=1, eps0=0.005, sigma_min=-4.5, sigma_max=-2.5,
                   DFL=0.1)
    qo, no, to, dto = O.timeloop(case, rp, 20)
    qg, ng, tg = run_gpu(dev, case, rp, 20, fused=fused)
    assert ng == no
    assert abs(tg - to) <= 1e-12 * to
    errs = fields_rel_l2(case, qg, qo)
    assert max(errs) <= 1e-12, errs


@pytest.mark.parametrize("fused", SCHEDULES, ids=SCHEDULE_IDS)
def test_flood_positivity(dev, fused):
    """Wet/dry flood on a curved 10x10 N=4 mesh with the positivity limiter."""
    case = Case.flood(N=4, nel=10, seed=1)
    rp = RunParams(num_flux=3, positivity=1, pos_pres_tol=1e-3, CFL=0.25)
    qo, no, to, _ = O.timeloop(case, rp, 20)
    qg, ng, tg = run_gpu(dev, case, rp, 20, fused=fused)
    assert ng == no
    errs = fields_rel_l2(case, qg, qo)
    assert max(errs) <= 1e-12, errs
    Q = qg.reshape(case.Nelem, 3, -1)
    assert np.isfinite(Q).all() and (Q[:, 0] >= 0).all()


@pytest.mark.parametrize("fused", SCHEDULES, ids=SCHEDULE_IDS)
def test_ocean_uplift_open_boundary(dev, fused):
    """Tsunami-like uplift over a 4000 m ocean with a shelf: open (still-water) boundary over the
    deep part, walls over the shelf, N=5 Cartesian 8x8, 30 steps."""
    case = Case.ocean_uplift(N=5, nel=8, amp=3.0, axis_a=80e3, axis_c=40e3, angle=0.6)
    rp = RunParams(num_flux=3, bc_kind=2, h_zero=4000.0)
    qo, no, to, _ = O.timeloop(case, rp, 30)
    qg, ng, tg = run_gpu(dev, case, rp, 30, fused=fused)
    assert ng == no == 30 and abs(tg - to) <= 1e-14 * to
    h, hu, hv = fields_rel_l2(case, qg, qo)
    assert max(h, hu, hv) <= 1e-12, (h, hu, hv)


@pytest.mark.parametrize("fused", SCHEDULES, ids=SCHEDULE_IDS)
@pytest.mark.parametrize("num_flux", [4, 5], ids=["roe", "ocean_combined"])
def test_roe_and_combined_ocean_flux(dev, fused, num_flux):
    """NumFlux 4 (Roe) and 5 (Roe on the open-ocean boundary, rotated ES elsewhere) over the ocean
    uplift with its open/wall boundary, 20 steps."""
    case = Case.ocean_uplift(N=4, nel=8, amp=3.0, axis_a=90e3, axis_c=70e3, angle=0.4)
    rp = RunParams(num_flux=num_flux, bc_kind=2, h_zero=4000.0)
    qo, no, to, _ = O.timeloop(case, rp, 20)
    qg, ng, tg = run_gpu(dev, case, rp, 20, fused=fused)
    assert ng == no == 20 and abs(tg - to) <= 1e-14 * to
    errs = fields_rel_l2(case, qg, qo)
    assert max(errs) <= 1e-12, errs


def test_manufactured_solution_parity_and_convergence(dev):
    """Convergence test (Dirichlet_ConvTest.okl + S_ConvTest.okl): the reference kernel sequence on
    the GPU against the oracle, and its error against the exact solution at order N+1."""
    from test_oracle_properties import manufactured
    case = Case.convergence(N=3, nel=6, curved=True)
    rp = RunParams(num_flux=3, bc_kind=3, CFL=0.2)
    qo, no, to, _ = O.timeloop(case, rp, 20)
    qg, ng, tg = run_gpu(dev, case, rp, 20, fused=0)
    assert ng == no and abs(tg - to) <= 1e-14 * to
    assert max(fields_rel_l2(case, qg, qo)) <= 1e-12
    errs = []
    for nel in (4, 8, 16):
        c = Case.convergence(N=3, nel=nel)
        rpT = RunParams(num_flux=0, bc_kind=3, CFL=0.2, T=0.2)
        q, n, t = run_gpu(dev, c, rpT, 100000, fused=0)
        assert t == 0.2
        errs.append(np.abs(q - manufactured(c, t)).max())
    eoc = np.log2(np.array(errs[:-1]) / np.array(errs[1:]))
    assert (eoc >= 3.7).all(), (errs, eoc)


@pytest.mark.parametrize("testcase,CFL", [(8, 0.2), (88, 0.2), (89, 0.01)])
def test_manufactured_variants_match_oracle(dev, testcase, CFL):
    """Testcases 8, 88, 89 (Dirichlet_ConvTest3/4/5.okl + S_ConvTest3/4/5.okl) on the curved mesh:
    the reference kernel sequence on the GPU against the oracle over 20 steps; the state stays
    within the discretisation error of the exact solution, whose time-dependent part has amplitude 1
    in h (the oracle's errors: 4e-3, 7e-4, 5e-3)."""
    from test_oracle_properties import manufactured
    case = Case.convergence(N=3, nel=6, curved=True, testcase=testcase)
    rp = RunParams(num_flux=0, bc_kind=S.CONVERGENCE_BC[testcase], CFL=CFL)
    qo, no, to, _ = O.timeloop(case, rp, 20)
    qg, ng, tg = run_gpu(dev, case, rp, 20, fused=0)
    assert ng == no == 20 and abs(tg - to) <= 1e-14 * to
    assert max(fields_rel_l2(case, qg, qo)) <= 1e-12
    assert np.abs(qg - manufactured(case, tg, testcase)).max() <= 0.02


def test_entropy_conservative_flux(dev):
    """ES=0 (EC surface flux): total entropy changes only by the time-integration error."""
    case = Case.gaussian_bump(N=4, nel=8)
    rp = RunParams(num_flux=0, ES=0, CFL=0.1)
    qg, _, _ = run_gpu(dev, case, rp, 50)
    dS = total_entropy(case, qg, rp.g) - total_entropy(case, case["q"], rp.g)
    rp1 = RunParams(num_flux=0, ES=1, CFL=0.1)
    qg1, _, _ = run_gpu(dev, case, rp1, 50)
    dS1 = total_entropy(case, qg1, rp.g) - total_entropy(case, case["q"], rp.g)
    assert abs(dS) < 1e-12
    assert dS1 < -1e-10


@pytest.mark.parametrize("av,pos", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_fused_equals_reference_sequence_bitwise(dev, av, pos):
    """The fused schedule performs the same arithmetic: identical state after 10 steps."""
    case = Case.dam_break(N=7, nel=8, noise=1e-3, seed=5) if not pos else Case.flood(N=5, nel=8, seed=2)
    rp = RunParams(num_flux=3, artificial_viscosity=av, eps0=0.005, sigma_min=-4.5, sigma_max=-2.5,
                   positivity=pos, pos_pres_tol=1e-3, CFL=0.25 if pos else 0.5)
    qa, na, ta = run_gpu(dev, case, rp, 10, fused=0)
    qb, nb, tb = run_gpu(dev, case, rp, 10, fused=1)
    assert na == nb and ta == tb
    assert np.array_equal(qa, qb) or np.abs(qa - qb).max() <= 1e-15 * np.abs(qa).max()


@pytest.mark.parametrize("av,pos", [(0, 0), (1, 0), (1, 1)])
def test_fused_update_evaluates_sensor_and_wave_speed(dev, av, pos):
    """The fused state update (with the limiter when it is on) also evaluates ShockCapturing (every
    stage) and FindLambdaMax (last stage) of the state it writes: after a run, ViscPara,
    ViscForPlot and LambdaMax equal those kernels applied to the final state, bit for bit."""
    case = Case.dam_break(N=7, nel=8, noise=1e-3, seed=5) if not pos else Case.flood(N=5, nel=8, seed=2)
    rp = RunParams(num_flux=3, artificial_viscosity=av, eps0=0.005, sigma_min=-4.5, sigma_max=-2.5,
                   positivity=pos, pos_pres_tol=1e-3, CFL=0.25 if pos else 0.5)
    E = case.Nelem
    ctx = dev.Context(dev.make_params(case, rp))
    try:
        s = dev.Solver(ctx, case, rp, fused=1)
        n, _ = s.run(6)
        assert n == 6
        lam = s.view("LambdaMax", E).download()
        visc = s.view("ViscPara", E).download()
        plot = s.view("ViscForPlot", E).download()
        q = s.get_q()
        s.close()
        dq, dB = ctx.array(q), ctx.array(case["b"])
        dV, dS = ctx.array(case["VdmInv"]), ctx.array(case["EleSizes"])
        dvisc, dplot, dlam = ctx.empty(E), ctx.empty(E), ctx.empty(E)
        ctx.find_lambda_max(E, dq, dlam)
        ctx.shock_capturing(E, dq, dB, dV, dS, dvisc, dplot)
        assert np.array_equal(lam, dlam.download()) and (lam > 0).all()
        if av:
            assert np.array_equal(visc, dvisc.download()) and np.array_equal(plot, dplot.download())
            assert (visc > 0).any() and (visc == 0).any()
    finally:
        ctx.close()


@pytest.mark.parametrize("nel", [2, 8])
def test_fused_every_element_viscous(dev, nel):
    """sigma_max below every element's sensor value: every element has viscosity, so the face pass
    lists all of them (the list is full) and the AV and viscous face passes run everywhere; the
    fused schedule still equals the reference sequence.  nel = 2: each element is its own
    neighbour's neighbour on several sides."""
    case = Case.dam_break(N=7, nel=nel, noise=1e-3, seed=5)
    rp = RunParams(num_flux=3, artificial_viscosity=1, eps0=0.002, sigma_min=-40.0, sigma_max=-39.0, CFL=0.5)
    visc = np.zeros(case.Nelem)
    O.call("shock_capturing", O.params(case, rp), case.Nelem, case["q"], case["b"], case["VdmInv"], visc, None)
    assert (visc == rp.eps0).all()
    qa, na, ta = run_gpu(dev, case, rp, 6, fused=0)
    qb, nb, tb = run_gpu(dev, case, rp, 6, fused=1)
    assert na == nb == 6 and ta == tb
    assert np.array_equal(qa, qb) or np.abs(qa - qb).max() <= 1e-15 * np.abs(qa).max()


@pytest.mark.parametrize("pos", [0, 1])
def test_single_kernel_equals_fused_bitwise(dev, pos):
    """The single-kernel stage (device dt, ping-pong state, graph replay) performs the fused
    schedule's arithmetic: identical state and time after 11 steps (odd: graph pairs + one eager)."""
    case = Case.dam_break(N=7, nel=8, noise=1e-3, seed=5) if not pos else Case.flood(N=5, nel=8, seed=2)
    rp = RunParams(num_flux=3, positivity=pos, pos_pres_tol=1e-3, CFL=0.25 if pos else 0.5)
    qa, na, ta = run_gpu(dev, case, rp, 11, fused=1)
    qb, nb, tb = run_gpu(dev, case, rp, 11, fused=2)
    assert na == nb == 11 and ta == tb
    assert np.array_equal(qa, qb)


@pytest.mark.parametrize("fused,analysis", [(0, 1), (1, 0), (1, 1)], ids=["sequence", "fused", "fused_analysis"])
def test_checkpoint_restart_continues_bitwise(dev, tmp_path, fused, analysis):
    """10 steps in one run equal 5 steps, a checkpoint, a restart in a new solver and 5 more steps:
    state, time and the analysis buffers bit for bit.  A solver of another size refuses the file."""
    case = Case.dam_break(N=7, nel=8, noise=1e-3, seed=5)
    rp = RunParams(num_flux=3, artificial_viscosity=1, eps0=0.005, sigma_min=-4.5, sigma_max=-2.5,
                   h_zero=1.5, maximum_elevation=analysis, arrival_times=analysis)
    E, n2 = case.Nelem, case.ngl ** 2
    ctx = dev.Context(dev.make_params(case, rp))
    try:
        a = dev.Solver(ctx, case, rp, fused=fused)
        a.run(10)
        qa, ta = a.get_q(), a.time()
        ma = a.view("MaximumElevation", E * n2).download() if analysis else None
        a.close()
        b = dev.Solver(ctx, case, rp, fused=fused)
        b.run(5)
        ck = tmp_path / "state.ckp"
        b.checkpoint(ck)
        b.close()
        c = dev.Solver(ctx, case, rp, fused=fused)
        c.restart(ck)
        n, _ = c.run(5)
        assert n == 5
        assert np.array_equal(c.get_q(), qa) and c.time() == ta
        if analysis:
            assert np.array_equal(c.view("MaximumElevation", E * n2).download(), ma)
        c.close()
    finally:
        ctx.close()
    other = Case.dam_break(N=7, nel=6, noise=1e-3, seed=5)
    ctx = dev.Context(dev.make_params(other, rp))
    try:
        d = dev.Solver(ctx, other, rp, fused=fused)
        with pytest.raises(dev.EsdgDeviceError, match="differ"):
            d.restart(ck)
        d.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("fused", [0, 1], ids=["host_clock", "device_clock"])
def test_invalid_time_step_is_reported(dev, fused):
    """CFL = 0 gives dt = 0, which DGtimeloop's check rejects: both time loops (dt read back every
    step, and dt on the device) report the error and leave the state as it was."""
    case = Case.gaussian_bump(N=4, nel=6)
    rp = RunParams(num_flux=0, CFL=0.0)
    ctx = dev.Context(dev.make_params(case, rp))
    try:
        s = dev.Solver(ctx, case, rp, fused=fused)
        with pytest.raises(dev.EsdgDeviceError, match="not positive and finite"):
            s.run(3)
        assert np.array_equal(s.get_q(), case["q"])
        s.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("fused,av", [(2, 0), (1, 0), (1, 1)], ids=["single_kernel", "fused", "fused_av"])
def test_device_clock_stops_at_T_and_resumes(dev, fused, av):
    """Device-side clock (the single-kernel stage, and the fused schedule without analysis buffers):
    steps issued after t reaches T change nothing and are not counted; a second run() continues
    from the first one's state and time."""
    case = Case.gaussian_bump(N=4, nel=8) if not av else Case.dam_break(N=7, nel=8, noise=1e-3, seed=5)
    extra = dict(artificial_viscosity=1, eps0=0.005, sigma_min=-4.5, sigma_max=-2.5, num_flux=3) if av else \
        dict(num_flux=0)
    rp_free = RunParams(**extra)
    _, _, t9 = run_gpu(dev, case, rp_free, 9, fused=0)
    _, _, t10 = run_gpu(dev, case, rp_free, 10, fused=0)
    rp = RunParams(**extra, T=0.5 * (t9 + t10))      # the 10th step is shortened to end at T
    qo, no, to, _ = O.timeloop(case, rp, 100)
    assert 10 <= no <= 11
    ctx = dev.Context(dev.make_params(case, rp))
    try:
        s = dev.Solver(ctx, case, rp, fused=fused)
        n1, t1 = s.run(7)
        n2, t2 = s.run(100)
        q = s.get_q()
        s.close()
    finally:
        ctx.close()
    assert n1 == 7 and n1 + n2 == no
    assert t1 < rp.T and t2 == to
    h, hu, hv = fields_rel_l2(case, q, qo)
    assert max(h, hu, hv) <= 1e-12, (h, hu, hv)


ISM_MESH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "meshes", "CircleInCircle.mesh")


@pytest.mark.parametrize("fused", SCHEDULES, ids=SCHEDULE_IDS)
def test_ism_mesh_bump_matches_oracle(dev, fused):
    """An ISM-V2 mesh with curved boundaries (the reference's CircleInCircle, 272 elements), N=4,
    walls, a Gaussian bump on the lake: 100 steps against the oracle."""
    case = Case.from_ism(ISM_MESH, N=4, case_kind=S.CASE_GAUSSIAN_BUMP, amp=0.05)
    rp = RunParams(num_flux=3)
    qo, no, to, _ = O.timeloop(case, rp, 100)
    qg, ng, tg = run_gpu(dev, case, rp, 100, fused=fused)
    assert ng == no == 100
    assert abs(tg - to) <= 1e-14 * to
    h, hu, hv = fields_rel_l2(case, qg, qo)
    assert h <= 1e-12 and hu <= 1e-12 and hv <= 1e-12, (h, hu, hv)


@pytest.mark.parametrize("N", [4, 6])
def test_ism_mesh_single_kernel_equals_fused_bitwise(dev, N):
    """On the curved ISM-V2 mesh (83 faces whose two sides run in opposite directions), at degrees
    whose line of nodes does not divide the wave (5 and 7 nodes), the single-kernel stage, which
    takes the reversed node's right trace from the lane holding it, equals the fused schedule,
    which evaluates each face once, bit for bit."""
    case = Case.from_ism(ISM_MESH, N=N, case_kind=S.CASE_GAUSSIAN_BUMP, amp=0.05)
    rp = RunParams(num_flux=3)
    qa, na, ta = run_gpu(dev, case, rp, 15, fused=1)
    qb, nb, tb = run_gpu(dev, case, rp, 15, fused=2)
    assert na == nb == 15 and ta == tb
    assert np.array_equal(qa, qb)


def test_ism_mesh_lake_at_rest(dev):
    """Lake at rest on the ISM mesh: the same state as the oracle's, and momentum bounded by what
    this mesh's geometry allows.  Its curved Coons patches preserve even a flat free stream only to
    about 6e-13 per step (oracle: 6e-11 after 100 steps with b = 0, the same with the bump); the
    Cartesian C0 mesh keeps 1e-13 (test_c0_lake_at_rest)."""
    case = Case.from_ism(ISM_MESH, N=4, case_kind=S.CASE_GAUSSIAN_BUMP, amp=0.0)
    rp = RunParams(num_flux=3)
    qg, ng, _ = run_gpu(dev, case, rp, 100, fused=1)
    qo, no, _, _ = O.timeloop(case, rp, 100)
    Q = qg.reshape(case.Nelem, 3, -1)
    assert np.abs(Q[:, 1]).max() <= 1e-9 and np.abs(Q[:, 2]).max() <= 1e-9
    assert np.abs(qg - qo).max() <= 1e-14


@pytest.mark.parametrize("learned", [False, True], ids=["sensor", "learned"])
def test_captured_fused_step_equals_eager(dev, learned):
    """From the second step of each run the fused schedule replays one captured step (dt, t and the
    stage marks live on the device; the marked-element update runs on the second stream inside the
    graph, and so does the learned indicator beside the face fluxes); a run with per-launch events
    stays eager, on one stream.  Both give the same bits over two run calls of 40 and 30 steps (a
    64-step chunk boundary inside), with the learned indicator's counts too."""
    case = Case.dam_break(N=7, nel=24, noise=1e-3, seed=7, ratio=2.5, angle=0.4)
    rp = RunParams(num_flux=3, artificial_viscosity=1, eps0=0.005, sigma_min=-4.5, sigma_max=-2.5, DFL=0.05)
    outs = []
    for prof in (False, True):
        ctx = dev.Context(dev.make_params(case, rp))
        try:
            s = dev.Solver(ctx, case, rp, fused=1)
            net = None
            if learned:
                net = dev.MLP(ctx, seed=3)
                s.set_indicator(net, 0.3, 0.7)
                s.indicator_audit(True)
            ctx.profile(prof)
            n1, _ = s.run(40)
            n2, t = s.run(30)
            q = s.get_q()
            counts = s.indicator_counts() if learned else None
            visc = s.view("ViscPara", case.Nelem).download()
            s.close()
            if net:
                net.close()
        finally:
            ctx.close()
        outs.append((q, n1 + n2, t, counts, visc))
    (qa, na, ta, ca, va), (qb, nb, tb, cb, vb) = outs
    assert (na, ta) == (nb, tb) == (70, tb)
    assert np.array_equal(qa, qb)
    assert ca == cb
    assert np.array_equal(va, vb)
    if not learned:
        assert (va > 0).any()


@pytest.mark.parametrize("fused", SCHEDULES, ids=SCHEDULE_IDS)
@pytest.mark.parametrize("N,av,pos", [(1, 0, 1), (2, 1, 0), (2, 1, 1)])
def test_lowest_degrees(dev, N, av, pos, fused):
    """Elements with fewer rows than the sensor's four energy sums and the limiter's three means."""
    if fused == 2 and N < 2:
        pytest.skip("the single-kernel stage starts at N = 2")
    case = Case.flood(N=N, nel=12, seed=4) if pos else Case.dam_break(N=N, nel=12, noise=1e-3, seed=4)
    rp = RunParams(num_flux=3, artificial_viscosity=av, eps0=0.005, sigma_min=-4.5, sigma_max=-2.5, DFL=0.05,
                   positivity=pos, pos_pres_tol=1e-3, CFL=0.1 if pos else 0.5)
    qo, no, to, _ = O.timeloop(case, rp, 6)
    qg, ng, tg = run_gpu(dev, case, rp, 6, fused=fused)
    assert ng == no == 6 and abs(tg - to) <= 1e-12 * to
    assert max(fields_rel_l2(case, qg, qo)) <= 1e-12


@pytest.mark.parametrize("av", [0, 1])
@pytest.mark.parametrize("mesh", ["affine", "affine_flat", "curved"])
@pytest.mark.parametrize("N", range(1, 10))
def test_fused_every_degree_equals_sequence_bitwise(dev, N, mesh, av):
    """Every degree of the fused schedule, and the single-kernel stage where it exists (2 <= N <= 7), on
    metrics and slopes from element records (affine_flat), metrics from records and slopes per node
    (affine), and everything per node (curved): state, time and the analysis buffers of 3 + 2 steps
    (each call an odd number) equal the reference sequence's, bit for bit."""
    if av and N == 1:
        pytest.skip("the sensor's two top shells need modes below them")
    if mesh == "curved":
        case, kw = Case.dam_break(N=N, nel=6, noise=1e-3, seed=N), dict(num_flux=3, h_zero=1.5)
    elif mesh == "affine":
        case, kw = Case.gaussian_bump(N=N, nel=6), dict(num_flux=0, h_zero=1.0)
    else:
        case, kw = Case.ocean_uplift(N=N, nel=6), dict(num_flux=3, bc_kind=2, h_zero=4000.0)
    q = case["q"].reshape(case.Nelem, 3, -1).copy()
    q[:, 0] *= 1.0 + 1e-3 * np.random.default_rng(N).uniform(-1.0, 1.0, q[:, 0].shape)
    case = case.with_state(q)
    rp = RunParams(artificial_viscosity=av, eps0=0.005, sigma_min=-4.5, sigma_max=-2.5, DFL=0.05, arrival_times=1,
                   maximum_elevation=1, **kw)
    size = case.Nelem * case.ngl ** 2
    outs = []
    for fused in (0, 1, 2):
        if fused == 2 and not 2 <= N <= 7:
            continue
        r = RunParams(**{**vars(rp), "arrival_times": int(fused < 2), "maximum_elevation": int(fused < 2)})
        ctx = dev.Context(dev.make_params(case, r))
        try:
            s = dev.Solver(ctx, case, r, fused=fused)
            n = s.run(3)[0] + s.run(2)[0]
            extra = [s.view(b, size).download() for b in ("ArrivalTimings", "MaximumElevation")] if fused < 2 else []
            outs.append((n, s.time(), s.get_q(), *extra))
            s.close()
        finally:
            ctx.close()
    ref = outs[0]
    assert ref[0] == 5 and np.isfinite(ref[2]).all()
    for o in outs[1:]:
        assert o[:2] == ref[:2]
        assert all(np.array_equal(a, b) for a, b in zip(o[2:], ref[2:]))


@pytest.mark.parametrize("av", [0, 1])
@pytest.mark.parametrize("fused", [1, 2])
def test_step_counts_of_either_parity(dev, fused, av):
    """The step's clock, maxima and marks alternate between two halves: calls of odd and even step counts, a
    call of no steps, and a new state between calls equal one run of the same steps, bit for bit."""
    case = Case.dam_break(N=4, nel=9, noise=1e-3, seed=6)
    rp = RunParams(num_flux=3, artificial_viscosity=av, eps0=0.005, sigma_min=-4.5, sigma_max=-2.5, DFL=0.05)
    ctx = dev.Context(dev.make_params(case, rp))
    try:
        a, b = dev.Solver(ctx, case, rp, fused=fused), dev.Solver(ctx, case, rp, fused=fused)
        assert a.run(9)[0] == 9
        assert [b.run(k)[0] for k in (1, 2, 0, 3, 1, 2)] == [1, 2, 0, 3, 1, 2]
        assert a.time() == b.time() and np.array_equal(a.get_q(), b.get_q())
        for s, parts in ((a, (4,)), (b, (3, 1))):
            s.set_q(case["q"])
            assert sum(s.run(k)[0] for k in parts) == 4
        assert np.array_equal(a.get_q(), b.get_q()) and a.last_dt() == b.last_dt()
        a.close()
        b.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("N,nel", [(2, 103), (2, 104), (4, 78), (4, 79), (5, 50), (5, 51), (7, 45), (7, 46), (7, 3)])
def test_wide_blocks_up_to_one_round(dev, N, nel):
    """Meshes on either side of the size up to which a block has five waves, and a mesh of one partly filled
    block: the state after three steps equals the reference sequence's, bit for bit."""
    case = Case.dam_break(N=N, nel=nel, noise=1e-3, seed=N)
    rp = RunParams(num_flux=3, artificial_viscosity=1, eps0=0.005, sigma_min=-4.5, sigma_max=-2.5, DFL=0.05)
    qa, na, ta = run_gpu(dev, case, rp, 3, fused=0)
    qb, nb, tb = run_gpu(dev, case, rp, 3, fused=1)
    assert na == nb == 3 and ta == tb
    assert np.array_equal(qa, qb)


def register_run(dev, case, rp, fused, calls, net=None, fails=False):
    """(steps, time, last dt, q, gRK) after the calls of run(), the last of which must fail with `fails`; `net`: (lo, hi)
    of a learned indicator."""
    ctx = dev.Context(dev.make_params(case, rp))
    try:
        s = dev.Solver(ctx, case, rp, fused=fused)
        mlp = dev.MLP(ctx, seed=1) if net else None
        if net:
            s.set_indicator(mlp, *net)
        n = 0
        for k in calls[:-1] if fails else calls:
            n += s.run(k)[0]
        if fails:
            with pytest.raises(dev.EsdgDeviceError, match="not positive and finite"):
                s.run(calls[-1])
        q = s.get_q()
        out = (n, s.time(), s.last_dt(), q, s.view("gRK", q.size).download())
        extra = [s.view(b, case.Nelem).download() for b in ("ViscPara", "ViscForPlot", "LambdaMax")]
        s.close()
        if mlp:
            mlp.close()
    finally:
        ctx.close()
    return out, extra


@pytest.mark.parametrize("end", ["odd", "even", "chunks", "T"])
@pytest.mark.parametrize("rk", [3, 4])
@pytest.mark.parametrize("fused,N,av", [(1, 1, 0), (1, 4, 0), (2, 4, 0), (1, 7, 1), (2, 7, 1), (1, 8, 1)])
def test_register_after_a_run(dev, fused, N, av, rk, end):
    """The low-storage RK register that a run leaves (buffer "gRK", which a checkpoint holds) is the reference
    sequence's, bit for bit: after odd and even step counts, more steps than are issued at a time, and a run that
    ends at T."""
    case = Case.dam_break(N=N, nel=5, noise=1e-3, seed=N)
    kw = dict(num_flux=3, rk_order=rk, artificial_viscosity=av, eps0=0.005, sigma_min=-4.5, sigma_max=-2.5, DFL=0.05, CFL=0.2)
    calls = dict(odd=(2, 3), even=(1, 4), chunks=(67,), T=(100,))[end]
    if end == "T":
        kw["T"] = 4.5 * run_gpu(dev, case, RunParams(**kw), 1)[2]
    rp = RunParams(**kw)
    ref = register_run(dev, case, rp, 0, calls)[0]
    got = register_run(dev, case, rp, fused, calls)[0]
    assert np.abs(ref[4]).max() > 0 and np.isfinite(ref[4]).all()
    assert got[:3] == ref[:3]
    assert np.array_equal(got[3], ref[3]) and np.array_equal(got[4], ref[4])


@pytest.mark.parametrize("split", [0, 1, 2])
@pytest.mark.parametrize("N,kind", [(4, "overflow"), (7, "overflow"), (7, "viscosity"), (7, "learned")])
def test_register_after_a_failed_step(dev, N, kind, split):
    """A run that ends because the next dt is not positive and finite leaves q and the RK register as the last good
    step left them, bit for bit, and the wave speeds and viscosities of that state: with a wave speed that has
    overflowed (no finite end time bounds dt), and with DFL = 0, which gives dt = 0 once an element has viscosity.
    split: steps taken by a first call, so that the failing step starts from either state buffer."""
    case = Case.gaussian_bump(N=N, nel=5)
    if kind == "overflow":
        rp = RunParams(num_flux=3, CFL=8.0, T=np.inf)
    else:
        rp = RunParams(num_flux=3, artificial_viscosity=1, eps0=0.005, sigma_min=-4.0, sigma_max=-2.0, DFL=0.0)
    ref, _ = register_run(dev, case, rp, 0, (split, 150), fails=True)
    got, extra = register_run(dev, case, rp, 1, (split, 150), net=(0.0, 1.0) if kind == "learned" else None, fails=True)
    assert ref[1] > 0 and (kind == "overflow" or np.isfinite(ref[4]).all() and np.abs(ref[4]).max() > 0)
    assert got[:3] == ref[:3]
    assert np.array_equal(got[3], ref[3], equal_nan=True)
    assert np.array_equal(got[4], ref[4], equal_nan=True)
    ctx = dev.Context(dev.make_params(case, rp))
    try:
        E = case.Nelem
        dq, lam, visc, plot = ctx.array(got[3]), ctx.empty(E), ctx.empty(E), ctx.empty(E)
        ctx.find_lambda_max(E, dq, lam)
        assert np.array_equal(extra[2], lam.download(), equal_nan=True)
        if rp.artificial_viscosity:
            ctx.shock_capturing(E, dq, ctx.array(case["b"]), ctx.array(case["VdmInv"]), ctx.array(case["EleSizes"]), visc, plot)
            assert np.array_equal(extra[0], visc.download()) and np.array_equal(extra[1], plot.download())
            assert (extra[0] > 0).any()
    finally:
        ctx.close()


@pytest.mark.parametrize("steps", [0, 2])
@pytest.mark.parametrize("ended", [False, True])
def test_single_kernel_viscosity_of_the_state(dev, ended, steps):
    """The single-kernel schedule leaves ViscPara and ViscForPlot of the state that a call ends with, also where the
    call takes no step: none asked for, or the end time reached."""
    case = Case.dam_break(N=4, nel=6, noise=1e-3, seed=3)
    rp = RunParams(num_flux=3, artificial_viscosity=1, eps0=0.005, sigma_min=-4.5, sigma_max=-2.5, DFL=0.05,
                   T=0.0 if ended else 1e30)
    ctx = dev.Context(dev.make_params(case, rp))
    try:
        E = case.Nelem
        s = dev.Solver(ctx, case, rp, fused=2)
        for q in (case["q"], 1.5 * case["q"].reshape(E, 3, -1)[::-1].ravel()):
            s.set_q(q)
            assert s.run(steps)[0] == (0 if ended else steps)
            dq, visc, plot = ctx.array(s.get_q()), ctx.empty(E), ctx.empty(E)
            ctx.shock_capturing(E, dq, ctx.array(case["b"]), ctx.array(case["VdmInv"]), ctx.array(case["EleSizes"]), visc, plot)
            assert (visc.download() > 0).any()
            assert np.array_equal(s.view("ViscPara", E).download(), visc.download())
            assert np.array_equal(s.view("ViscForPlot", E).download(), plot.download())
        s.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("fused", SCHEDULES, ids=SCHEDULE_IDS)
@pytest.mark.parametrize("mesh", ["affine", "curved"])
def test_bottom_traces_written_between_runs(dev, mesh, fused):
    """The buffers "bL" and "bR" are the bottom traces that the face fluxes read: what a program writes there between
    two calls counts in the second, also where a Cartesian mesh's face geometry comes from records."""
    case = Case.ocean_uplift(N=4, nel=6) if mesh == "affine" else Case.dam_break(N=4, nel=6, noise=1e-3, seed=2)
    rp = RunParams(num_flux=3, **(dict(bc_kind=2, h_zero=4000.0) if mesh == "affine" else {}))
    add = 0.01 * np.arange(case.Nfaces)[:, None] * (1.0 + np.outer(np.arange(case.Nfaces) % 2, np.arange(case.ngl)))
    outs = []
    for change in (False, True):
        for f in (0, fused):
            ctx = dev.Context(dev.make_params(case, rp))
            try:
                s = dev.Solver(ctx, case, rp, fused=f)
                bufs = [s.view(b, case.Nfaces * case.ngl) for b in ("bL", "bR")]
                s.run(2)
                if change:
                    for b in bufs:
                        v = b.download() + add.ravel() / case.Nfaces
                        ctx.check(dev.lib().esdg_memcpy(ctx.handle, ctypes.c_void_p(b.ptr), v.ctypes.data_as(ctypes.c_void_p),
                                                        v.nbytes, dev.ESDG_H2D))
                s.run(2)
                outs.append(s.get_q())
                s.close()
            finally:
                ctx.close()
    assert np.array_equal(outs[0], outs[1]) and not np.array_equal(outs[0], outs[2])
    assert np.array_equal(outs[2], outs[3])


@pytest.mark.parametrize("late", [False, True])
@pytest.mark.parametrize("calls", [(2,), (3,), (2, 3, 0)], ids=["even", "odd", "calls"])
@pytest.mark.parametrize("N,av", [(2, 0), (4, 1), (7, 1), (8, 0)])
def test_fused_face_buffers(dev, N, av, calls, late):
    """The fused schedule's buffers "FStar" and "Traces", which programs can ask for before a run or after it: the
    numerical fluxes of the last stage's state (the reference sequence's SurfaceParts) and the side traces of the
    state, in face slots.  (Asked for after an odd number of steps, FStar starts with the next call.)"""
    case = Case.dam_break(N=N, nel=6, noise=1e-3, seed=N)
    rp = RunParams(num_flux=3, artificial_viscosity=av, eps0=0.005, sigma_min=-4.5, sigma_max=-2.5, DFL=0.05)
    n, F = case.ngl, case.Nfaces
    ctx = dev.Context(dev.make_params(case, rp))
    try:
        a, s = dev.Solver(ctx, case, rp, fused=0), dev.Solver(ctx, case, rp, fused=1)
        if not late:
            s.view("FStar", F * 3 * n), s.view("Traces", F * 6 * n)
        for k in calls:
            assert a.run(k)[0] == s.run(k)[0] == k
        tr, fs = s.view("Traces", F * 6 * n).download().reshape(F, 2, 3, n), s.view("FStar", F * 3 * n).download()
        q = s.get_q().reshape(case.Nelem, 3, n * n)
        assert np.array_equal(q.ravel(), a.get_q())
        k = np.arange(n)
        node = np.stack([k, (k + 1) * n - 1, n * n - n + k, k * n])
        E = case["EdgeData"].reshape(F, 8)
        for f in range(F):
            for side in (0, 1):
                if E[f, 5 + side] == 0:
                    assert np.array_equal(tr[f, side], q[E[f, side]][:, node[E[f, 2 + side]]]), (f, side)
        if not (late and sum(calls) % 2):
            assert np.array_equal(fs, a.view("SurfaceParts", F * 3 * n).download())
        a.close()
        s.close()
    finally:
        ctx.close()


REFUSED = """
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)     # before the library: its calls bind here first
import numpy as np
import esdgsem_mpiocca_amd as E
dev = E.device()
case = E.Case.dam_break(N=4, nel=6, noise=1e-3, seed=2)
rp = E.RunParams(num_flux=3, artificial_viscosity=1, eps0=0.005, sigma_min=-4.5, sigma_max=-2.5, DFL=0.05)
ctx = dev.Context(dev.make_params(case, rp))
outs = []
for fused in (0, 1, 2):
    s = dev.Solver(ctx, case, rp, fused=fused)
    outs.append((s.run(3)[0] + s.run(20)[0], s.time(), s.get_q()))
    s.close()
ens = dev.Ensemble(ctx, [(case, rp, None)])
ens.run(23)
outs.append((ens.status(0)[1], ens.status(0)[0], ens.get_q(0)))
ens.close()
ctx.close()
assert ctypes.c_int.in_dll(shim, "refused").value == 3
assert all(o[:2] == outs[0][:2] and np.array_equal(o[2], outs[0][2]) for o in outs)
print("same states")
"""


@pytest.mark.parametrize("call", ["int hipStreamBeginCapture(void* s, int mode) { return ++refused, 900; }",
                                  "int hipGraphInstantiate(void** e, void* g, void** n, char* l, unsigned long k) { return ++refused, 2; }"],
                         ids=["begin", "instantiate"])
def test_refused_graph_capture_runs_eagerly(tmp_path, call):
    """Where the runtime refuses to capture steps or to instantiate the graph, they are launched one by one: the same
    states and times.  (In a process of its own, with that one call of the runtime replaced by a refusal.)"""
    src, lib = tmp_path / "refuse.c", tmp_path / "librefuse.so"
    src.write_text("int refused = 0;\n" + call + "\n")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src)], check=True)
    r = subprocess.run([sys.executable, "-c", REFUSED, str(lib)], capture_output=True, text=True, timeout=100,
                       cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert r.returncode == 0 and "same states" in r.stdout, r.stdout + r.stderr


@pytest.mark.parametrize("fused", [1, 2])
def test_steps_after_the_end_write_nothing(dev, fused):
    """Steps issued after t has reached T leave the state, which both buffers hold by then, without writing it again: a
    launch of theirs takes a sixth of a stage's time (carrying the state over in every stage took a third)."""
    case = Case.gaussian_bump(N=7, nel=256, build=False)
    us, outs = [], []
    for T in (1e30, 1e-9):
        rp = RunParams(num_flux=3, T=T)
        ctx = dev.Context(dev.make_params(case, rp))
        try:
            mesh = dev.DeviceCase(ctx, case)
            s = dev.Solver(ctx, mesh, rp, fused=fused)
            q0 = s.get_q()
            s.run(1)
            s.set_q(q0)
            ctx.profile(True)
            ctx.profile_reset()
            n, t = s.run(4 if T > 1 else 64)
            launches, ms = ctx.profile_query("stage")
            assert (n, launches) == ((4, 20) if T > 1 else (1, 320))
            us.append(ms / launches * 1e3)
            outs.append((t, s.get_q(), q0))
            s.close()
            mesh.close()
        finally:
            ctx.close()
    assert outs[1][0] == 1e-9 and np.abs(outs[1][1] - outs[1][2]).max() < 1e-6
    assert us[1] < 0.25 * us[0], us


@pytest.mark.parametrize("av", [0, 1])
@pytest.mark.parametrize("mesh", ["slopes", "flat"])
@pytest.mark.parametrize("N,nel", [(2, 103), (2, 104), (3, 6), (4, 78), (4, 79), (5, 7), (6, 6), (7, 45), (7, 46)])
def test_element_records_around_one_round(dev, N, nel, mesh, av):
    """Cartesian meshes, whose metrics come from element records (the slopes too where the bottom is flat), on either
    side of the size up to which a block has five waves, with and without viscosity: both fused schedules' state, register
    and viscosity equal the reference sequence's, bit for bit."""
    if mesh == "slopes":
        case, kw = Case.gaussian_bump(N=N, nel=nel), dict(num_flux=0)
    else:
        case, kw = Case.ocean_uplift(N=N, nel=nel), dict(num_flux=3, bc_kind=2, h_zero=4000.0)
    q = case["q"].reshape(case.Nelem, 3, -1).copy()
    rng = np.random.default_rng(N)
    rough = rng.uniform(size=(case.Nelem, 1)) < 0.3       # the others stay smooth
    q[:, 0] *= 1.0 + 1e-3 * rough * rng.uniform(-1.0, 1.0, q[:, 0].shape)
    case = case.with_state(q)
    rp = RunParams(artificial_viscosity=av, eps0=0.005, sigma_min=-9.0, sigma_max=-5.0, DFL=0.05, CFL=0.2, **kw)
    outs = []
    for fused in (0, 1, 2):
        ctx = dev.Context(dev.make_params(case, rp))
        try:
            s = dev.Solver(ctx, case, rp, fused=fused)
            n, t = s.run(3)
            visc = s.view("ViscPara", case.Nelem).download()
            outs.append((n, t, s.get_q(), s.view("gRK", q.size).download(), visc))
            s.close()
        finally:
            ctx.close()
    ref = outs[0]
    assert ref[0] == 3 and np.isfinite(ref[2]).all()
    assert not av or (ref[4] > 0).any() and (ref[4] == 0).any()
    for o in outs[1:]:
        assert o[:2] == ref[:2] and np.array_equal(o[2], ref[2]) and np.array_equal(o[3], ref[3])
    assert np.array_equal(outs[1][4], outs[2][4])


@pytest.mark.parametrize("av", [0, 1])
@pytest.mark.parametrize("fused,N", [(0, 4), (1, 4), (2, 4), (1, 8)])
def test_first_run_allocates_nothing(dev, fused, N, av):
    """All device memory of a solver is allocated with it: no run pays for an allocation, the first one included."""
    case = Case.dam_break(N=N, nel=6, noise=1e-3, seed=2)
    rp = RunParams(num_flux=3, artificial_viscosity=av, eps0=0.005, sigma_min=-4.5, sigma_max=-2.5, DFL=0.05)
    ctx = dev.Context(dev.make_params(case, rp))
    try:
        s = dev.Solver(ctx, case, rp, fused=fused)
        before = ctx.bytes_allocated()
        assert s.run(3)[0] == 3 and s.run(12)[0] == 12
        assert ctx.bytes_allocated() == before
        s.close()
    finally:
        ctx.close()

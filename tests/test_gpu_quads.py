"""The lane groups of the sweeps (four lanes per cell, 16 cells per wave) and
of the limiter (16 lanes per cell) at their edges, against the oracle: cell
counts around a group, a wave and a workgroup's worth of cells, the counts
where the workgroup size changes, and more limited cells than the limiter's
grid holds at once.  All of it is FP64 in the oracle's operation order, so the
tolerance is that of the other FP64 parity tests."""
# The Jacobi sweeps below run with 16 lanes per cell (k_jacobi_wide: A^-1 B up
# to 168 MB, here 58333 quads), the two largest and the mixed mesh with
# four (k_jacobi); a sweep's 256-thread workgroups, the FP32 sweep's and SOR's,
# are in test_gpu_sweep_variants.py.
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _case(kind, nx, ny, sor=0, limiter=0, seed=3, top=None):
    from dnds_amd import _capi as A
    from dnds_amd.host import RIEMANN_VR_SETTING, CompactFacedMeshSerialRW, VRFiniteVolume2D, vr_setting
    bcs = (A.BC_FARFIELD, A.BC_WALL_NOSLIP, A.BC_WALL_EULER, A.BC_WALL if top is None else top)
    mesh = CompactFacedMeshSerialRW.generate(kind, nx, ny, 0.0, 1.0, 0.0, ny / nx, jitter=0.2, seed=seed, bc=bcs)
    vfv = VRFiniteVolume2D(mesh, vr_setting(**dict(RIEMANN_VR_SETTING, far_weight=1.0, jacobi_relax=0.9),
                                            build_limiter_data=limiter, sor_instead=sor))
    vfv.Initialization(8)
    return mesh, vfv


def _state(n, seed):
    rng = np.random.default_rng(seed)
    rho, vx, vy, p = 1 + 0.3 * rng.random(n), 0.4 * rng.random(n), -0.3 * rng.random(n), 1 + 0.2 * rng.random(n)
    u = np.stack([rho, rho * vx, rho * vy, p / 0.4 + 0.5 * rho * (vx * vx + vy * vy)], 1)
    return u, 1e-2 * rng.standard_normal((n, 36))


def _oracle(mesh, vfv, far):
    import oracle
    st = vfv.setting
    return oracle.Oracle(mesh.arrays(), vfv.arrays(), riemann_solver=2, far_field=far, jacobi_relax=st.jacobi_relax,
                         tang_weight=st.tang_weight, tang_weight_direction=st.tang_weight_direction,
                         wbap_smooth_indicator_scale=st.wbap_smooth_indicator_scale)


FAR = (1.1, 0.3, -0.1, 2.8)


@pytest.mark.parametrize("kind,nx,ny", [(0, 1, 1), (1, 3, 5), (1, 4, 4), (1, 17, 1), (0, 4, 8), (1, 5, 13), (2, 9, 11),
                                        (1, 273, 274), (1, 274, 274), (2, 224, 224)])
def test_sweep_at_group_and_workgroup_edges(kind, nx, ny):
    from dnds_amd.host import EulerEvaluator
    mesh, vfv = _case(kind, nx, ny)
    ev = EulerEvaluator(mesh, vfv, riemannSolverType="HLLC", farFieldStaticValue=FAR)
    u, x = _state(mesh.n_cell, 5)
    du, dx, dn = ev.BuildMean().upload(u), vfv.BuildRec().upload(x), vfv.BuildRec()
    vfv.ReconstructionJacobiStep(du, dx, dn, 0.0)
    ref = _oracle(mesh, vfv, FAR).jacobi_step(u, x)
    assert rel_err(dn.download(), ref) <= TOL
    assert rel_err(dx.download(), ref) <= TOL
    ev.device.sync()


@pytest.mark.parametrize("procedure", [2, 3])
def test_more_limited_cells_than_the_grid_holds(procedure):
    from dnds_amd.host import EulerEvaluator
    mesh, vfv = _case(2, 304, 304, limiter=1)  # about 138 000 cells, 131 072 at once
    assert mesh.n_cell > 131072
    ev = EulerEvaluator(mesh, vfv, riemannSolverType="HLLC", farFieldStaticValue=FAR)
    u, x = _state(mesh.n_cell, 6)
    du, dx, dn = ev.BuildMean().upload(u), vfv.BuildRec().upload(x), vfv.BuildRec()
    limit = vfv.ReconstructionWBAPLimitFacialV3 if procedure == 3 else vfv.ReconstructionWBAPLimitFacialV2
    limit(du, dx, dn, ifAll=True)
    orc = _oracle(mesh, vfv, FAR)
    ref, _ = (orc.wbap_v3 if procedure == 3 else orc.wbap_v2)(u, x, if_all=True)
    assert rel_err(dn.download(), ref) <= TOL


@pytest.mark.parametrize("nx,ny,sor", [(1, 1, 0), (5, 51, 0), (16, 16, 0), (257, 1, 0), (64, 64, 0), (241, 17, 1),
                                       (300, 300, 0)])
def test_sweep_increment_at_sum_edges(nx, ny, sor):
    """The increment that ReconstructToTolerance returns, (1 / n) sum over
    cells of |x_new - x_old|^2, from cell counts around a tree of 256 and a
    workgroup of 16 trees, with both workgroup sizes of the sweep and with
    SOR: sums of positive terms in FP64, so 1e-12 holds for any order."""
    from dnds_amd.host import EulerEvaluator
    mesh, vfv = _case(1, nx, ny, sor=sor)
    ev = EulerEvaluator(mesh, vfv, riemannSolverType="HLLC", farFieldStaticValue=FAR)
    u, x = _state(mesh.n_cell, 8)
    du, dx, dn = ev.BuildMean().upload(u), vfv.BuildRec().upload(x), vfv.BuildRec()
    before = x
    for _ in range(2):
        sweeps, increment = vfv.ReconstructToTolerance(du, dx, dn, 0.0, 1)
        new = dx.download()
        ref = ((new - before) ** 2).sum() / mesh.n_cell
        assert sweeps == 1 and abs(increment - ref) <= 1e-12 * ref
        before = new


@pytest.mark.parametrize("mu", [0.0, 1e-3])
@pytest.mark.parametrize("kind,nx,ny", [(1, 1, 1), (2, 7, 9), (1, 140, 141), (1, 141, 142), (0, 115, 116),
                                        (2, 127, 129)])
def test_rhs_face_quads_and_lanes(kind, nx, ny, mu):
    """EvaluateRHS on both sides of the face count (40000) where the face
    fluxes go from a quad per face to a lane per face, with far-field and wall
    boundaries in the same launch; one mixed step for the FP32 variant
    (its tolerance: FP32 sweeps and fluxes, as in the mixed-precision tests)."""
    import oracle
    from dnds_amd.host import EulerEvaluator, ExplicitSSPRK3LocalDt
    from dnds_amd import _capi as A
    mesh, vfv = _case(kind, nx, ny, top=A.BC_FARFIELD)
    assert (mesh.arrays()["face2cell"].size // 2 < 40000) == \
        (nx < 115 or (kind, nx) == (1, 140))
    u, x = _state(mesh.n_cell, 9)
    x = 0.1 * x
    ev = EulerEvaluator(mesh, vfv, riemannSolverType="HLLC", farFieldStaticValue=FAR, muGas=mu)
    st = vfv.setting
    orc = oracle.Oracle(mesh.arrays(), vfv.arrays(), riemann_solver=2, far_field=FAR, jacobi_relax=st.jacobi_relax,
                        tang_weight=st.tang_weight, tang_weight_direction=st.tang_weight_direction, mu_gas=mu)
    du, dx, rhs, dt = ev.BuildMean().upload(u), vfv.BuildRec().upload(x), ev.BuildMean(), ev.BuildScalar()
    ev.EvaluateDt(dt, du, CFL=0.5, MaxDt=1e100, UseLocaldt=True)
    ev.EvaluateRHS(rhs, du, dx, 0.1)
    _, _, _, dlf = orc.evaluate_dt(u, 0.5, use_local_dt=True)
    assert rel_err(rhs.download(), orc.evaluate_rhs(u, x, dlf, t=0.1)) <= TOL
    if mu == 0.0:
        r, rn = vfv.BuildRec().upload(x), vfv.BuildRec()
        ExplicitSSPRK3LocalDt(ev, nInternalRecStep=2, CFL=0.3, mixedPrecision=True).Step(du, r, rn, 0.0)
        ru, _, _ = orc.ssprk3_steps(u, x, 1, 2, 0.3)
        assert rel_err(du.download(), ru) <= 1e-6


@pytest.mark.parametrize("n", [240, 243])
def test_sweeps_on_both_sides_of_the_wide_one(n):
    """The last mesh whose sweep takes 16 lanes per cell (168 MB of A^-1 B) and
    one beyond it, with walls of every kind and the increment; then one
    mixed-precision step on far field and walls (tolerances as in its tests)."""
    from dnds_amd import _capi as A
    from dnds_amd.host import EulerEvaluator, ExplicitSSPRK3LocalDt
    mesh, vfv = _case(1, n, n)
    assert (4 * mesh.n_cell * 720 <= 168e6) == (n == 240)
    ev = EulerEvaluator(mesh, vfv, riemannSolverType="HLLC", farFieldStaticValue=FAR)
    u, x = _state(mesh.n_cell, 5)
    du, dx, dn = ev.BuildMean().upload(u), vfv.BuildRec().upload(x), vfv.BuildRec()
    _, increment = vfv.ReconstructToTolerance(du, dx, dn, 0.0, 1)
    ref = _oracle(mesh, vfv, FAR).jacobi_step(u, x)
    assert rel_err(dx.download(), ref) <= TOL
    expect = ((ref - x) ** 2).sum() / mesh.n_cell
    assert abs(increment - expect) <= 1e-11 * expect
    mesh, vfv = _case(1, n, n, top=A.BC_FARFIELD)
    ev = EulerEvaluator(mesh, vfv, riemannSolverType="HLLC", farFieldStaticValue=FAR)
    du, dx, dn = ev.BuildMean().upload(u), vfv.BuildRec().upload(0.1 * x), vfv.BuildRec()
    ExplicitSSPRK3LocalDt(ev, nInternalRecStep=2, CFL=0.3, mixedPrecision=True).Step(du, dx, dn, 0.0)
    ru, rr, _ = _oracle(mesh, vfv, FAR).ssprk3_steps(u, 0.1 * x, 1, 2, 0.3)
    assert rel_err(du.download(), ru) <= 1e-6 and rel_err(dx.download(), rr) <= 1e-5

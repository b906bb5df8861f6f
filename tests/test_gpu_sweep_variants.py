"""Sweeps on meshes past the sizes where another kernel, workgroup or cache
policy takes over, against the oracle:

* the Jacobi sweep goes from 16 lanes per cell (k_jacobi_wide) to four
  (k_jacobi) where the A^-1 B stream (720 bytes per cell and face) exceeds
  168 MB, and then keeps only a share of the stream in the cache;
* the FP32 correction sweep (336 bytes per cell and face) and an SOR colour
  take workgroups of 256 threads instead of 64 from 300000 lanes (75000
  cells) on; the former keeps a share of its stream beyond 168 MB, and the
  FP64 sweep of a mixed step keeps none beyond 450 MB.

FP64 sweeps run in the oracle's operation order, so the tolerance is that of
the other FP64 parity tests; mixed steps have that of the mixed-precision
tests (FP32 rounding of the corrections, 1e-5 of the coefficients and 1e-6 of
the means after one step)."""
import numpy as np
import pytest

from conftest import rel_err
from test_gpu_quads import FAR, TOL, _case, _oracle, _state

pytestmark = pytest.mark.gpu


def _pairs(mesh):
    """(cell, face) pairs of the mesh"""
    return int(np.diff(mesh.arrays()["cell_ptr"]).sum())


# triangles and mixed cells past 168 MB (a kept share of 41 and 39 blocks of
# 64), then past 168 MB of FP32 stream, then past 450 MB of FP64 stream; no
# cell count is a multiple of 64
@pytest.mark.parametrize("kind,nx,ny,kept32,kept64", [(0, 199, 201, True, True), (2, 223, 227, True, True),
                                                      (0, 287, 299, False, True), (0, 331, 333, False, False)])
def test_four_lane_sweeps_and_their_mixed_step(kind, nx, ny, kept32, kept64):
    from dnds_amd import _capi as A
    from dnds_amd.host import EulerEvaluator, ExplicitSSPRK3LocalDt
    mesh, vfv = _case(kind, nx, ny, top=A.BC_FARFIELD)
    n, pairs = mesh.n_cell, _pairs(mesh)
    assert n % 64 and 720 * pairs > 168e6 and 4 * n >= 300000
    assert (336 * pairs <= 168e6) == kept32 and (720 * pairs <= 450e6) == kept64
    ev = EulerEvaluator(mesh, vfv, riemannSolverType="HLLC", farFieldStaticValue=FAR)
    orc = _oracle(mesh, vfv, FAR)
    u, x = _state(n, 12)
    x = 0.1 * x
    du, dx, dn = ev.BuildMean().upload(u), vfv.BuildRec().upload(x), vfv.BuildRec()
    vfv.ReconstructionJacobiStep(du, dx, dn, 0.0)
    assert rel_err(dx.download(), orc.jacobi_step(u, x)) <= TOL
    dx.upload(x)
    ode = ExplicitSSPRK3LocalDt(ev, nInternalRecStep=4, CFL=0.3, mixedPrecision=True)
    dt = ode.Step(du, dx, dn, 0.0)
    ru, rx, rt = orc.ssprk3_steps(u, x, 1, 4, 0.3)
    assert abs(dt - rt) <= TOL * rt
    assert rel_err(du.download(), ru) <= 1e-6 and rel_err(dx.download(), rx) <= 1e-5


@pytest.mark.parametrize("kind,nx,ny", [(0, 303, 307), (1, 403, 391)])
def test_sor_colours_of_256_thread_workgroups(kind, nx, ny):
    """Two sweeps over colours of more than 75000 cells whose ranges do not
    start on a group of 16."""
    from dnds_amd.host import EulerEvaluator
    mesh, vfv = _case(kind, nx, ny, sor=1)
    ev = EulerEvaluator(mesh, vfv, riemannSolverType="HLLC", farFieldStaticValue=FAR)
    colour, n_colour = ev.LUSGSColouring()
    size = np.bincount(colour, minlength=n_colour)
    assert size.max() >= 75000 and np.any(np.cumsum(size)[:-1] % 16)
    u, x = _state(mesh.n_cell, 13)
    du, dx, dn = ev.BuildMean().upload(u), vfv.BuildRec().upload(x), vfv.BuildRec()
    orc, scan, ref = _oracle(mesh, vfv, FAR), ev.LUSGSScanOrder(), x
    for _ in range(2):
        vfv.ReconstructionJacobiStep(du, dx, dn, 0.0)
        ref = orc.sor_step(u, ref, scan)
        assert rel_err(dx.download(), ref) <= TOL
    ev.device.sync()

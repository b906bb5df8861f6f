"""Device arrays hold the host's values exactly, whatever the device's
numbering: cell counts around a block of 64, cell kinds sorted within the
blocks (mixed meshes) and colour-major numbering (SOR_Instead)."""
import numpy as np
import pytest

from test_gpu_quads import FAR, _case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,nx,ny,sor", [(1, 1, 1, 0), (1, 9, 7, 0), (1, 8, 8, 0), (1, 13, 5, 0), (2, 31, 17, 0),
                                            (0, 40, 23, 1), (2, 60, 47, 1)])
def test_upload_download_round_trip(kind, nx, ny, sor):
    from dnds_amd.host import EulerEvaluator
    mesh, vfv = _case(kind, nx, ny, sor=sor)
    ev = EulerEvaluator(mesh, vfv, riemannSolverType="HLLC", farFieldStaticValue=FAR)
    for a in (vfv.BuildRec(), ev.BuildMean(), ev.BuildScalar()):
        h = np.random.default_rng(mesh.n_cell).standard_normal(a.shape())
        a.upload(h)
        assert np.array_equal(a.download(), h)
        # the rest of the last block is no part of the array: a constant, then
        # the same rows again
        a.setConstant(3.0).upload(h[::-1].copy())
        assert np.array_equal(a.download(), h[::-1])


def test_a_failed_allocation_is_reported_once():
    """A warm start for 10^10 training rows (2.3 TB) is refused; the calls
    after it are not."""
    from conftest import rel_err
    from dnds_amd import _capi as A
    from dnds_amd.host import DNDSError, EulerEvaluator, WarmStart
    from test_gpu_quads import TOL, _oracle, _state
    mesh, vfv = _case(1, 12, 9)
    ev = EulerEvaluator(mesh, vfv, riemannSolverType="HLLC", farFieldStaticValue=FAR)
    u, x = _state(mesh.n_cell, 4)
    du, dx, dn = ev.BuildMean().upload(u), vfv.BuildRec().upload(x), vfv.BuildRec()
    with pytest.raises(DNDSError) as e:
        WarmStart(ev, capacity=10**10)
    assert e.value.code == A.ERR_OUT_OF_MEMORY
    vfv.ReconstructionJacobiStep(du, dx, dn, 0.0)
    assert rel_err(dx.download(), _oracle(mesh, vfv, FAR).jacobi_step(u, x)) <= TOL
    ev.device.sync()

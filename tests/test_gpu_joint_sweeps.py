"""The joint launches of small grids (face fluxes, EMF sweeps and face
velocities by block range; boundary work likewise) against the one-face-per-
thread kernels in launches of their own: the same expressions, so every array
must be bit-identical. Sizes: the smallest grid, fewer shells than the outer
boundary's EMF blend touches, k-rows below and above the row kernel's limit
of 24 faces, tiles ending inside an axis and just after it, and one size above
the joint launches' limit (1,000,000 cells)."""
import numpy as np
import pytest

from conftest import bits_equal, gcs_config, problem

pytestmark = pytest.mark.gpu

CHECKED = (problem.STATE_FIELDS + [problem.EDGE_EMF + d for d in range(3)]
           + [problem.FLUID_FACE_FLUX + d for d in range(3)]
           + [problem.MAXWELL_FACE_FLUX + d for d in range(3)])


@pytest.mark.parametrize("nr,n,mi", [(2, 9, False), (3, 10, False), (16, 12, True),
                                     (7, 16, False), (5, 23, False), (9, 33, False),
                                     (71, 49, False)])
def test_joint_launches_bitwise_equal_plain_kernels(gpu, nr, n, mi):
    cfg = gcs_config.earth_problem(nr, n, perturbation=0.01, seed=nr + n, mi=mi, mi_azimuth=32,
                                   mi_colatitude=12, outer_radius=30.0 if nr > 4 else 4.0)
    print(f"joint sweeps {nr} x {n}^2", flush=True)
    a, b = gpu.GpuProblem(cfg), gpu.GpuProblem(cfg)
    a.set_graph(True)
    b.set_plain_kernels(True)
    for _ in range(3):
        a.advance(1)
        b.advance(1)
        assert a.clock() == b.clock()
    for fid in CHECKED:
        for f in range(gcs_config.FACE_COUNT):
            x = a.field(f, fid)
            assert np.isfinite(x).all() and bits_equal(x, b.field(f, fid)), (fid, f)

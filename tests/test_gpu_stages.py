"""The stage table of profiled steps (time_steps): it times the launches that
an unprofiled step runs, and every stage it names is one that some step has."""
import pytest

from conftest import bits_equal, gcs_config, problem

pytestmark = pytest.mark.gpu

EVERY = {"ghost_fill", "earth_ghosts", "predict", "earth_emf", "sync_edges", "update",
         "finish_step", "seam_recover"}
DIRECTIONS = {f"{s}_{d}" for s in ("face_flux", "edge_emf") for d in "ijk"}
# first steps (a CFL pass, a recovery of every cell), and ends of steps
ONCE = {"cfl", "earth_recover", "mi_update", "end"}


@pytest.mark.parametrize("nr,n,mixed,plain,sweeps", [
    (16, 12, False, False, {"sweeps", "sweeps_end"}),
    (71, 49, False, False, DIRECTIONS | {"finish_flux", "face_velocity"}),
    (16, 12, False, True, DIRECTIONS | {"finish_flux", "face_velocity"}),
    (16, 12, True, False, {"face_flux", "edge_emf", "finish_flux", "face_velocity"}),
])
def test_stages_are_those_of_the_step(gpu, nr, n, mixed, plain, sweeps):
    cfg = gcs_config.earth_problem(nr, n, perturbation=0.01, seed=2)
    a, b = gpu.GpuProblem(cfg), gpu.GpuProblem(cfg)
    for p in (a, b):
        p.set_fidelity(False)
        p.set_plain_kernels(plain)
        p.set_precision(mixed)
        p.advance(2)
    total, stages = a.time_steps(3)
    b.advance(3)
    timed = {k for k, v in stages.items() if v > 0.0}
    print(nr, n, mixed, plain, sorted(timed), flush=True)
    assert timed == EVERY | sweeps
    # (event times are floats)
    assert sum(stages.values()) <= 1.001 * total
    assert set(stages) == EVERY | ONCE | DIRECTIONS | {
        "face_flux", "edge_emf", "finish_flux", "face_velocity", "sweeps", "sweeps_end"}
    for fid in (problem.CONSERVED, problem.FACE_FLUX):
        assert bits_equal(a.field(0, fid), b.field(0, fid))

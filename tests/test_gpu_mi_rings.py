"""The register-resident polar solves (one wavefront per colatitude ring) at
the sizes where their layout can go wrong: one ring and one point per lane up
to eight, rings that end inside a lane, exactly full workgroups (six rings)
and one ring more.

The current of a generated potential (gcs_problem_mi_make_pairs) is solved
from zero and must give that potential back. Tolerance: the solve stops at a
residual of 1e-12 of the right-hand side, and the error is at most the
operator's condition times that; the smallest eigenvalue of the polar
operator is of order one of its colatitude coupling, and the largest, the
longitude coupling of the ring next to the pole, exceeds it by less than 1e3
(the residual norm weighs that ring up by the same sine), so 1e-9 of the
largest potential is the bound. The single-workgroup solve of the same
problem (GCS_MI_COOPERATIVE=0, read when a problem is made) must agree to
twice that."""
import importlib

import numpy as np
import pytest

from conftest import gcs_config

pytestmark = pytest.mark.gpu

TOL = 1e-9


@pytest.mark.parametrize("hall", [0.0, 5.0])
@pytest.mark.parametrize("nt,np_", [(3, 8), (4, 64), (8, 65), (9, 57), (14, 130), (20, 200),
                                    (15, 256), (26, 321), (13, 385), (10, 449), (33, 512)])
def test_ring_solves_return_the_generated_potential(gpu, monkeypatch, nt, np_, hall):
    ws = importlib.import_module("gamera-cube_amd.warm_start")
    cfg = gcs_config.earth_problem(16, 12, mi=True, hall_siemens=hall, mi_azimuth=np_,
                                   mi_colatitude=nt)
    cfg.mi.relative_tolerance = 1e-12
    print(f"ring solve {nt} x {np_} hall {hall}", flush=True)
    p = gpu.GpuProblem(cfg)
    cur, pot = ws.make_pairs(p, seed=nt + np_, count=2, pedersen=cfg.mi.pedersen_siemens,
                             hall=hall)
    scale = np.abs(pot).max()
    got, cold, _ = ws.solve_current(p, cur, np.zeros_like(pot), use_network=False)
    print(f"  iterations {cold}, error {np.abs(got - pot).max() / scale:.1e}", flush=True)
    assert np.abs(got - pot).max() <= TOL * scale
    # from the solution itself: no more iterations than from zero (a BiCGStab
    # solve may have stopped on its recursive residual, with the true one a
    # little above the bound, so a few can be left), the same potential
    again, warm, _ = ws.solve_current(p, cur, got, use_network=False)
    assert sum(warm) <= sum(cold) and np.abs(again - got).max() <= TOL * scale
    monkeypatch.setenv("GCS_MI_COOPERATIVE", "0")
    q = gpu.GpuProblem(cfg)
    single, _, _ = ws.solve_current(q, cur, np.zeros_like(pot), use_network=False)
    assert np.abs(single - got).max() <= 2 * TOL * scale


# Colatitude points up to the most that one wavefront per ring can take (128
# workgroups a hemisphere, two on 256 compute units), and one more.
RING_LIMIT = 770


@pytest.mark.parametrize("nt,np_", [(400, 9), (RING_LIMIT, 64), (RING_LIMIT + 1, 64)])
@pytest.mark.parametrize("hall", [0.0, 5.0])
def test_solves_of_many_rings(gpu, monkeypatch, nt, np_, hall):
    """Reductions over more than 64 workgroups (67 and 128 a hemisphere), and
    the Hall solve beyond the ring kernel's limit, which must still be spread
    over the chip: several times faster an iteration than one workgroup per
    hemisphere (by 8 and more when measured).

    Tolerance: a residual of 1e-12 of the right-hand side bounds the error by
    1e-12 times the ratio of the right-hand side to the potential, and that
    grows with the longitude coupling of the ring next to the pole, 1 /
    sin(theta)^2, as the square of the rings' number: TOL, which holds to 33
    rings, times (nt / 33)^2."""
    ws = importlib.import_module("gamera-cube_amd.warm_start")
    cfg = gcs_config.earth_problem(16, 12, mi=True, hall_siemens=hall, mi_azimuth=np_,
                                   mi_colatitude=nt)
    cfg.mi.relative_tolerance = 1e-12
    tol = TOL * (nt / 33) ** 2

    def solve():
        p = gpu.GpuProblem(cfg)
        cur, pot = ws.make_pairs(p, seed=nt + np_, count=2, pedersen=cfg.mi.pedersen_siemens,
                                 hall=hall)
        got, its, ms = ws.solve_current(p, cur, np.zeros_like(pot), use_network=False)
        scale = np.abs(pot).max()
        err = np.abs(got - pot).max() / scale
        print(f"  {nt} x {np_} hall {hall}: iterations {its}, {ms:.1f} ms, error {err:.1e}",
              flush=True)
        assert err <= tol
        return got / scale, ms / max(its)

    spread, spread_ms = solve()
    monkeypatch.setenv("GCS_MI_COOPERATIVE", "0")
    single, single_ms = solve()
    assert np.abs(single - spread).max() <= 2 * tol
    if hall > 0.0 and np_ == 64:
        assert spread_ms < 0.5 * single_ms


@pytest.mark.parametrize("hall", [0.0, 5.0])
@pytest.mark.parametrize("polls", [1, 50])
def test_solve_after_a_wait_that_was_given_up(gpu, monkeypatch, polls, hall):
    """A wait between workgroups that runs out of its polls (GCS_MI_SPIN_LIMIT,
    read when a problem is made) must not end the solve: one workgroup per
    hemisphere solves the system. One poll never suffices for all six
    workgroups of each of a hundred iterations, so there the bits are those of
    that solve asked first; 50 may or may not."""
    ws = importlib.import_module("gamera-cube_amd.warm_start")
    cfg = gcs_config.earth_problem(16, 12, mi=True, hall_siemens=hall, mi_azimuth=65,
                                   mi_colatitude=33)
    cfg.mi.relative_tolerance = 1e-12
    monkeypatch.setenv("GCS_MI_COOPERATIVE", "0")
    p = gpu.GpuProblem(cfg)
    cur, pot = ws.make_pairs(p, seed=3, count=2, pedersen=cfg.mi.pedersen_siemens, hall=hall)
    guess = 0.5 * pot
    single, its, _ = ws.solve_current(p, cur, guess, use_network=False)
    monkeypatch.delenv("GCS_MI_COOPERATIVE")
    monkeypatch.setenv("GCS_MI_SPIN_LIMIT", str(polls))
    q = gpu.GpuProblem(cfg)
    scale = np.abs(pot).max()
    for _ in range(2):
        got, got_its, _ = ws.solve_current(q, cur, guess, use_network=False)
        if polls == 1:
            assert got_its == its and np.array_equal(got, single)
        assert np.abs(got - pot).max() <= TOL * scale
    # and in a coupled run
    q.advance(2)
    assert q.mi_report()["ready"] and np.isfinite(q.mi_field(0)).all()

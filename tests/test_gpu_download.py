"""Downloads of whole-plane fields: interleaved on the device, fetched for all
cube faces at once below 4 MiB and one face at a time above, in chunks that
end inside a face. Two problems in the same state that download in opposite
orders (one after an earlier download that a step made stale) must give the
same arrays bit for bit, and the face frames must equal those inside the cell
geometry, which another path lays out.
"""
import ctypes

import numpy as np
import pytest

from conftest import bits_equal, gcs_config, problem

pytestmark = pytest.mark.gpu

FIELDS = [f for f in range(problem.FIELD_COUNT)
          if f not in (problem.HYDRO_RATE, problem.MAXWELL_RATE)]


@pytest.mark.parametrize("nr,n", [(2, 9), (16, 12), (40, 30), (96, 40)])
def test_downloads_do_not_depend_on_their_order(gpu, nr, n):
    cfg = gcs_config.earth_problem(nr, n, perturbation=0.01, seed=5,
                                   outer_radius=30.0 if nr > 4 else 4.0)
    a, b = gpu.GpuProblem(cfg), gpu.GpuProblem(cfg)
    a.advance(1)
    a.field(5, problem.CONSERVED)  # stale after the next step
    a.advance(1)
    b.advance(2)
    first = {(f, fid): a.field(f, fid).copy() for fid in FIELDS for f in range(6)}
    for f in reversed(range(6)):
        for fid in reversed(FIELDS):
            x = b.field(f, fid)
            assert bits_equal(x, first[f, fid]), (f, fid)
    ni, nj, nk = cfg.extent
    for f in (0, 5):
        cell = first[f, problem.CELL_GEOMETRY].reshape(ni, nj, nk, 103)
        for d in range(3):
            ext = [ni, nj, nk]
            ext[d] += 1
            face = first[f, problem.FACE_GEOMETRY + d].reshape(*ext, 16)
            lower = cell[..., 4 + 32 * d:4 + 32 * d + 16]
            assert np.array_equal(lower, face[:ni, :nj, :nk])


def test_download_on_a_full_device(gpu):
    """A face's geometry (278 MB) with less than 200 MB left on the device."""
    lib = gpu.library()  # the HIP runtime's symbols are those of its dependency

    def left():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    p = gpu.GpuProblem(gcs_config.earth_problem(192, 96, perturbation=0.01, seed=5))
    fields = [problem.FACE_GEOMETRY, problem.CONSERVED]
    p.advance(1)
    hold = []
    while left() > 192 << 20:
        hold.append(ctypes.c_void_p())
        assert lib.hipMalloc(ctypes.byref(hold[-1]),
                             ctypes.c_size_t(left() - (160 << 20))) == 0
    print(f"{left() >> 20} MiB left", flush=True)
    full = [p.field(f, fid).copy() for fid in fields for f in (0, 5)]
    for h in hold:
        assert lib.hipFree(h) == 0
    p.advance(1)  # drops the geometry's host arrays
    q = gpu.GpuProblem(p.config)
    q.advance(1)
    again = [q.field(f, fid) for fid in fields for f in (0, 5)]
    assert all(bits_equal(a, b) for a, b in zip(full, again))
    # the same problem goes back to the interleaved path
    assert all(bits_equal(p.field(f, problem.FACE_GEOMETRY), a) for f, a in zip((0, 5), full))

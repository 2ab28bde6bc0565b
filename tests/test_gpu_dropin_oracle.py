"""The drop-in entry points against the oracle's six-face step (bitwise the
reference's, tests/test_oracle_vs_reference.py), with no reference at hand: a
caller's grid, storage and background of include/gamera_cs_types.h, filled from
the library's own problem, stepped by gamera_cs_advance_six_with_background_
planned and by orc_advance_six on two copies.

The drop-in runs its step in four phases with host work possible between them,
so its launches are others than those of a problem's step: the ghost fill by
itself, the sweeps never joined, boundary work switched by the callbacks given.
Cases: the Earth callbacks recognised by address (device kernels), the same
with an ionosphere of the library, callbacks at other addresses (run on the
host between the phases), no boundary at all (radial outflow), hydrodynamic
steps, five ghost layers, and resident storage.

Tolerance: as tests/test_dropin.py, 1e-13 a step on |a - b| / max(1, |a|), from
the last digits of ROCm's transcendental functions."""
import ctypes

import numpy as np
import pytest

from conftest import gcs_config, problem
from test_dropin import STEP_TOL, WRITTEN, worst

pytestmark = pytest.mark.gpu

VP, SZ, D = ctypes.c_void_p, ctypes.c_size_t, ctypes.c_double
B, I = ctypes.c_bool, ctypes.c_int
SZ3 = SZ * 3


class FaceGrid(ctypes.Structure):
    _fields_ = [("extent", SZ3), ("value", VP)]


class EdgeGrid(ctypes.Structure):
    _fields_ = [("extent", SZ3), ("value", VP), ("valid", VP)]


class Grid(ctypes.Structure):
    _fields_ = [("cell_extent", SZ3), ("vertex_extent", SZ3), ("vertex", VP), ("cell", VP),
                ("face", FaceGrid * 3), ("edge", EdgeGrid * 3)]


class Storage(ctypes.Structure):
    _fields_ = [("cell_extent", SZ3), ("face_extent", SZ3 * 3), ("edge_extent", SZ3 * 3),
                ("conserved", VP), ("old_conserved", VP), ("predicted_conserved", VP),
                ("cell_magnetic", VP), ("old_cell_magnetic", VP), ("predicted_cell_magnetic", VP),
                ("face_flux", VP * 3), ("old_face_flux", VP * 3), ("predicted_face_flux", VP * 3),
                ("edge_emf", VP * 3), ("fluid_face_flux", VP * 3), ("maxwell_face_flux", VP * 3),
                ("hydro_rate", VP), ("maxwell_rate", VP),
                ("emergency_diffusion_face_count", SZ),
                ("emergency_diffusion_max_interface_speed", D),
                ("inner_wall_clamped_face_count", SZ * 2),
                # the other inner-wall statistics: 13 pairs of doubles and one of vectors
                ("inner_wall", D * (2 * 13 + 6))]


class Background(ctypes.Structure):
    _fields_ = [("cell_magnetic", VP), ("face_magnetic", VP * 3), ("face_flux", VP * 3),
                ("edge_magnetic", VP * 3), ("cell_force", VP)]


class Sweep(ctypes.Structure):
    _fields_ = ([(n, D) for n in ("gamma", "density_floor", "pressure_floor", "pdm", "hydro_hogs",
                                  "magnetic_hogs", "light_speed")]
                + [(n, B) for n in ("use_mhd", "use_hogs", "use_boris", "use_background")])


class Emf(ctypes.Structure):
    _fields_ = ([(n, D) for n in ("density_floor", "pdm", "diffusion", "light_speed", "cfl", "dt")]
                + [(n, B) for n in ("use_boris", "use_background")])


class Update(ctypes.Structure):
    _fields_ = ([(n, D) for n in ("gamma", "density_floor", "pressure_floor", "light_speed")]
                + [(n, B) for n in ("use_mhd", "use_boris", "use_background")])


class Options(ctypes.Structure):
    _fields_ = [("stress", Sweep), ("emf", Emf), ("update", Update), ("cell_source", VP),
                ("source_context", VP), ("indexed_cell_source", VP),
                ("indexed_source_context", VP), ("source_time", D), ("fluid_flux_sync", VP),
                ("fluid_flux_context", VP), ("edge_emf_sync", VP), ("edge_emf_context", VP)]


class WindState(ctypes.Structure):
    _fields_ = [("density", D), ("pressure", D), ("velocity", D * 3), ("magnetic", D * 3)]


class Wind(ctypes.Structure):
    _fields_ = [("count", SZ), ("time", VP), ("state", VP), ("reference", D * 3),
                ("time_offset", D), ("by", D), ("bz", D), ("bx", D), ("enforce_bx", I),
                ("linear", I)]


class Boundary(ctypes.Structure):
    _fields_ = [("startup", VP), ("wind", VP), ("background", VP), ("mi", VP),
                ("density_floor", D), ("pressure_floor", D), ("step_time", D), ("step_dt", D),
                ("cfl", D), ("strict_inner_gas_wall", I)]


class StepContext(ctypes.Structure):  # orc_step_context
    _fields_ = [("halo", VP), ("edges", VP), ("earth", VP), ("mi", VP)]


# the callback types of include/gamera_cs_types.h
RADIAL = ctypes.CFUNCTYPE(I, VP, VP, VP, SZ, D, D, VP)
SYNC = ctypes.CFUNCTYPE(I, VP, VP, VP, VP, VP)


class Caller:
    """A program's arrays and contexts for one problem, copied from `source`;
    `field` reads them as test_dropin.worst does."""

    def __init__(self, source, cfg, background=True, mhd=True):
        ce = list(cfg.extent)
        ve = [e + 1 for e in ce]
        fe = [[e + (a == d) for a, e in enumerate(ce)] for d in range(3)]
        ee = [[e + (a != d) for a, e in enumerate(ce)] for d in range(3)]
        self.keep = [[source.field(f, fid).copy() for fid in range(problem.FIELD_COUNT)]
                     for f in range(6)]
        for f in range(6):  # zero until a step writes them
            for fid in set(WRITTEN) - set(problem.STATE_FIELDS):
                self.keep[f][fid][:] = 0.0
        self.valid = [[source.edge_valid(f, d).copy() for d in range(3)] for f in range(6)]
        self.grid, self.storage, self.background = (Grid * 6)(), (Storage * 6)(), (Background * 6)()
        for f in range(6):
            def at(fid, f=f):
                return self.keep[f][fid].ctypes.data
            g, s, b = self.grid[f], self.storage[f], self.background[f]
            g.cell_extent = s.cell_extent = SZ3(*ce)
            g.vertex_extent = SZ3(*ve)
            g.vertex, g.cell = at(problem.VERTEX), at(problem.CELL_GEOMETRY)
            for name, fid in (("conserved", problem.CONSERVED),
                              ("old_conserved", problem.OLD_CONSERVED),
                              ("predicted_conserved", problem.PREDICTED_CONSERVED),
                              ("cell_magnetic", problem.CELL_MAGNETIC),
                              ("old_cell_magnetic", problem.OLD_CELL_MAGNETIC),
                              ("predicted_cell_magnetic", problem.PREDICTED_CELL_MAGNETIC),
                              ("hydro_rate", problem.HYDRO_RATE),
                              ("maxwell_rate", problem.MAXWELL_RATE)):
                setattr(s, name, at(fid))
            b.cell_magnetic, b.cell_force = at(problem.BG_CELL_MAGNETIC), at(problem.BG_CELL_FORCE)
            for d in range(3):
                g.face[d].extent, g.face[d].value = SZ3(*fe[d]), at(problem.FACE_GEOMETRY + d)
                g.edge[d].extent, g.edge[d].value = SZ3(*ee[d]), at(problem.EDGE_GEOMETRY + d)
                g.edge[d].valid = self.valid[f][d].ctypes.data
                s.face_extent[d], s.edge_extent[d] = SZ3(*fe[d]), SZ3(*ee[d])
                for name, fid in (("face_flux", problem.FACE_FLUX),
                                  ("old_face_flux", problem.OLD_FACE_FLUX),
                                  ("predicted_face_flux", problem.PREDICTED_FACE_FLUX),
                                  ("edge_emf", problem.EDGE_EMF),
                                  ("fluid_face_flux", problem.FLUID_FACE_FLUX),
                                  ("maxwell_face_flux", problem.MAXWELL_FACE_FLUX)):
                    getattr(s, name)[d] = at(fid + d)
                b.face_magnetic[d] = at(problem.BG_FACE_MAGNETIC + d)
                b.face_flux[d] = at(problem.BG_FACE_FLUX + d)
                b.edge_magnetic[d] = at(problem.BG_EDGE_MAGNETIC + d)
        self.active = SZ3(cfg.radial_cells, cfg.angular_cells, cfg.angular_cells)
        self.ghost = cfg.ghost
        su, boris = cfg.startup, bool(cfg.use_boris)
        # the serial Earth driver's options (test_cubedsphere_dipole_background.c:405-449)
        self.options = Options(
            stress=Sweep(su.gamma, 1e-6, 1e-8, 1.0, 0.25, 0.25, 10.0, mhd, True, boris,
                         background),
            emf=Emf(1e-6, 1.0, 0.5, 10.0, cfg.cfl, 0.0, boris, background),
            update=Update(su.gamma, 1e-6, 1e-8, 10.0, mhd, boris, background))
        pressure = su.density * su.speed ** 2 / (su.gamma * su.mach ** 2)
        self.wind_time = (D * 1)(cfg.wind_time[0])
        self.wind_state = (WindState * 1)(WindState(su.density, pressure, (su.speed, 0.0, 0.0),
                                                    tuple(su.imf.value)))
        self.wind = Wind(count=1, time=ctypes.addressof(self.wind_time),
                         state=ctypes.addressof(self.wind_state), linear=1,
                         reference=(cfg.wind_reference_x, 0.0, 0.0))
        self.startup = su
        self.boundary = Boundary(startup=ctypes.addressof(su), wind=ctypes.addressof(self.wind),
                                 background=ctypes.addressof(self.background),
                                 density_floor=1e-6, pressure_floor=1e-8, cfl=cfg.cfl,
                                 strict_inner_gas_wall=cfg.strict_inner_gas_wall)

    def field(self, f, fid):
        return self.keep[f][fid]

    def counters(self, f):
        s = self.storage[f]
        return s.emergency_diffusion_face_count, s.emergency_diffusion_max_interface_speed


class OracleStepper:
    def __init__(self, orc, caller, earth, mi_cfg=None):
        for name in ("orc_halo_plan_build", "orc_edge_plan_build"):
            fn = getattr(orc, name)
            fn.restype, fn.argtypes = VP, [VP, VP, SZ]
        orc.orc_halo_plan_free.argtypes = orc.orc_edge_plan_free.argtypes = [VP]
        orc.orc_advance_six.argtypes = [VP, VP, VP, SZ, D, D, VP, VP, VP, D, D]
        self.orc, self.c, self.mi = orc, caller, VP()
        self.context = StepContext(
            halo=orc.orc_halo_plan_build(caller.grid, caller.active, caller.ghost),
            edges=orc.orc_edge_plan_build(caller.grid, caller.active, caller.ghost),
            earth=ctypes.addressof(caller.boundary) if earth else None)
        if mi_cfg is not None:
            orc.orc_mi_create.argtypes = [VP, VP, VP, VP, VP, SZ, VP, D, VP]
            orc.orc_mi_maybe_update.argtypes = [VP, D]
            assert orc.orc_mi_create(caller.grid, caller.storage, caller.background,
                                     ctypes.addressof(caller.startup), caller.active,
                                     caller.ghost, ctypes.byref(mi_cfg), 0.0,
                                     ctypes.byref(self.mi)) == 0
            self.context.mi = self.mi
            caller.boundary.mi = self.mi

    def step(self, ratio, dt, t, t_prev):
        c = self.c
        if self.mi:
            assert self.orc.orc_mi_maybe_update(self.mi, t) >= 0
        c.boundary.step_time, c.boundary.step_dt = t, dt
        assert self.orc.orc_advance_six(
            c.grid, c.storage, c.active, c.ghost, ratio, dt, ctypes.byref(c.options),
            c.background, ctypes.byref(self.context), t, t_prev) == 0

    def close(self):
        if self.mi:
            self.orc.orc_mi_destroy.argtypes = [VP]
            self.orc.orc_mi_destroy(self.mi)
        self.orc.orc_halo_plan_free(self.context.halo)
        self.orc.orc_edge_plan_free(self.context.edges)


class DropinStepper:
    """callbacks: "device" (addresses the library recognises; never called),
    "host" (the oracle's boundary functions at other addresses), or None."""

    def __init__(self, gpu, orc, caller, callbacks, mi_cfg=None):
        lib = self.lib = gpu.library()
        self.gpu, self.c, self.mi = gpu, caller, VP()
        lib.gamera_cs_advance_six_with_background_planned.argtypes = [
            VP, VP, VP, SZ, D, D, VP, VP, VP, VP, D, D, VP]
        lib.gcs_dropin_release.argtypes = [VP, VP]
        lib.gcs_dropin_sync_to_host.argtypes = [VP, VP]
        lib.gcs_dropin_host_round_trips.restype = ctypes.c_long
        lib.gcs_dropin_register_earth_callbacks.argtypes = [VP, VP, VP]
        never = (RADIAL(lambda *a: -1), SYNC(lambda *a: -1), SYNC(lambda *a: -1))
        lib.gcs_dropin_register_earth_callbacks(*[ctypes.cast(f, VP) for f in never])
        self.radial, self.functions = None, [never]
        if callbacks == "host":
            orc.orc_earth_ghosts.argtypes = [VP, VP, VP, SZ, D, D, VP, VP]
            orc.orc_earth_inner_flux.argtypes = [VP, VP, VP]
            orc.orc_earth_emf.argtypes = [VP, VP, VP, VP, VP, VP]
            own = (RADIAL(lambda g, s, a, n, t, tp, ctx:
                          orc.orc_earth_ghosts(g, s, a, n, t, tp, ctx, None)),
                   SYNC(lambda s, g, lo, hi, ctx: orc.orc_earth_inner_flux(s, lo, hi)),
                   SYNC(lambda s, g, lo, hi, ctx: orc.orc_earth_emf(s, g, lo, hi, ctx, None)))
            self.functions.append(own)
        if callbacks is not None:
            f = [ctypes.cast(x, VP) for x in self.functions[-1]]
            self.radial = f[0]
            caller.options.fluid_flux_sync, caller.options.edge_emf_sync = f[1], f[2]
            caller.options.edge_emf_context = ctypes.addressof(caller.boundary)
        if mi_cfg is not None:
            lib.gamera_cs_mi_dipole_create.argtypes = [VP, VP, VP, VP, VP, SZ, VP, VP]
            lib.gamera_cs_mi_dipole_maybe_update.argtypes = [VP, D]
            assert lib.gamera_cs_mi_dipole_create(
                caller.grid, caller.storage, caller.background,
                ctypes.addressof(caller.startup), caller.active, caller.ghost,
                ctypes.byref(mi_cfg), ctypes.byref(self.mi)) == 0
            caller.boundary.mi = self.mi

    def step(self, ratio, dt, t, t_prev):
        c = self.c
        if self.mi:
            assert self.lib.gamera_cs_mi_dipole_maybe_update(self.mi, t) >= 0
        c.boundary.step_time, c.boundary.step_dt = t, dt
        rc = self.lib.gamera_cs_advance_six_with_background_planned(
            c.grid, c.storage, c.active, c.ghost, ratio, dt, ctypes.byref(c.options),
            c.background if c.options.update.use_background else None, None, self.radial, t,
            t_prev, ctypes.byref(c.boundary))
        assert rc == 0, self.gpu.last_error()

    def close(self):
        if self.mi:
            self.lib.gamera_cs_mi_dipole_destroy.argtypes = [VP]
            self.lib.gamera_cs_mi_dipole_destroy(self.mi)
        self.lib.gcs_dropin_release(self.c.grid, self.c.storage)
        self.lib.gcs_dropin_register_earth_callbacks(None, None, None)


@pytest.mark.parametrize("name,steps,callbacks,mhd,mi,resident", [
    ("small", 6, "device", True, False, False),
    ("ragged", 4, "device", True, False, True),
    ("ghost5", 4, "device", True, False, False),
    ("fast_wind", 4, "device", True, False, False),
    ("small", 4, "device", False, False, False),
    ("small", 3, "host", True, False, False),
    ("small", 4, None, True, False, False),
    ("ragged", 4, None, False, False, False),
    ("small_mi", 6, "device", True, True, False),
])
def test_dropin_matches_oracle(gpu, orc, name, steps, callbacks, mhd, mi, resident):
    cfg = gcs_config.workload(name)
    cfg.mi.relative_tolerance = 1e-13
    source = gpu.GpuProblem(cfg)
    background = callbacks is not None
    a = Caller(source, cfg, background, mhd)
    b = Caller(source, cfg, background, mhd)
    source.advance(1)
    dt = 0.5 * source.clock()["dt"]
    source.close()
    oracle = OracleStepper(orc, a, callbacks is not None, cfg.mi if mi else None)
    dropin = DropinStepper(gpu, orc, b, callbacks, cfg.mi if mi else None)
    rounds = gpu.library().gcs_dropin_host_round_trips()
    gpu.library().gcs_dropin_set_resident(1 if resident else 0)
    try:
        t = 0.0
        for s in range(steps):
            ratio, t_prev = (0.0, t) if s == 0 else (0.5, t - dt)
            oracle.step(ratio, dt, t, t_prev)
            dropin.step(ratio, dt, t, t_prev)
            if resident:
                assert gpu.library().gcs_dropin_sync_to_host(b.grid, b.storage) == 0
            t += dt
            err, where = worst(a, b)
            print(f"drop-in {name} {callbacks} mhd {mhd} mi {mi} step {s + 1}: {err:.2e} at "
                  f"{where}", flush=True)
            assert err <= STEP_TOL * (s + 1), where
            for f in range(6):
                ca, cb = a.counters(f), b.counters(f)
                assert ca[0] == cb[0] and abs(ca[1] - cb[1]) <= 1e-12 * max(1.0, ca[1])
        moved = gpu.library().gcs_dropin_host_round_trips() - rounds
        assert moved == (3 * steps if callbacks == "host" else 0)
    finally:
        gpu.library().gcs_dropin_set_resident(0)
        dropin.close()
        oracle.close()
    assert gpu.library().gcs_dropin_mirror_count() == 0

"""Performance cases: what a user of this package has the GPU do.

Three paths, each through the package's public entry points:

* "step": a six-face Earth problem (`native.GpuProblem`) advances a batch of
  driver steps and the state is read back (`advance`, `field`, `clock`), the
  cycle of a run between two output frames.
* "polar": one ionosphere potential solve of both hemispheres
  (`warm_start.solve_current`), from the potential of the last update.
* "unet": the learned warm start's network: `forward`, `gradients`, and the
  training loop (`warm_start.train`).

Sizes are those of the repository's workloads (`config.workload`), tests and
benchmark, plus odd and ragged ones between them.
"""
import importlib
import math

import numpy as np
import torch

_cfg = importlib.import_module("gamera-cube_amd.config")
_native = importlib.import_module("gamera-cube_amd.native")
_problem = importlib.import_module("gamera-cube_amd.problem")
_ws = importlib.import_module("gamera-cube_amd.warm_start")

# Compulsory bytes of one FP64 cell update: 30 state and 122 geometry and
# background doubles, each once. The mixed form's compulsory bytes are taken
# as the same, as it keeps the FP64 state.
STEP_BYTES = 1216
# FP64 operations of one cell update, counted as about 2,000 a face and edge
# pair per direction.
STEP_FLOPS = 6000

PEDERSEN = 10.0
HALL = 5.0
# The network's 3x3 convolutions (cin, cout), in parameter order.
LAYERS = [(32, 32), (32, 32), (32, 64), (64, 64), (64, 128), (128, 128), (128, 256), (256, 256),
          (384, 128), (128, 128), (192, 64), (64, 64), (96, 32), (32, 32)]
LEVEL = [0, 0, 1, 1, 2, 2, 3, 3, 2, 2, 1, 1, 0, 0]


def listed():
    return [
        # The smallest coupled run of the tests, with the package's default
        # options: every kernel launched by itself, ghost values of the
        # storage reproduced, a Pedersen solve on a 32 x 12 polar grid about
        # once a pass. Latency and launches count.
        {"name": "step_small_coupled", "kind": "step", "nr": 16, "n": 12, "steps": 40,
         "mixed": False, "fidelity": True, "graph": False, "nt": 12, "np": 32, "hall": 0.0},
        # config0 (6 x 24^2 x 48) with the default options.
        {"name": "step_config0", "kind": "step", "nr": 48, "n": 24, "steps": 20,
         "mixed": False, "fidelity": True, "graph": False, "nt": 0, "np": 0, "hall": 0.0},
        # A medium grid with odd extents, where every tile and block range is
        # partial; the benchmark's options (graph launches, no ghost upkeep).
        {"name": "step_ragged", "kind": "step", "nr": 75, "n": 45, "steps": 20,
         "mixed": False, "fidelity": False, "graph": True, "nt": 0, "np": 0, "hall": 0.0},
        # The mixed form (FP32 reconstruction, fluxes and EMF) at half of
        # config1's resolution.
        {"name": "step_mixed", "kind": "step", "nr": 96, "n": 48, "steps": 40,
         "mixed": True, "fidelity": False, "graph": True, "nt": 0, "np": 0, "hall": 0.0},
        # config1 (6 x 96^2 x 192, ionosphere on 2 x 128 x 256, Hall 5 S)
        # with the benchmark's options: the headline run.
        {"name": "step_config1", "kind": "step", "nr": 192, "n": 96, "steps": 40,
         "mixed": False, "fidelity": False, "graph": True, "nt": 128, "np": 256, "hall": HALL},
        # config1's ionosphere update: the Hall-tensor solve.
        {"name": "polar_hall_config1", "kind": "polar", "nt": 128, "np": 256, "hall": HALL},
        # The same grids without a Hall conductance (the default of
        # `earth_problem(mi=True)`): the Pedersen solve.
        {"name": "polar_pedersen", "kind": "polar", "nt": 128, "np": 256, "hall": 0.0},
        # A small polar grid with odd extents.
        {"name": "polar_hall_odd", "kind": "polar", "nt": 33, "np": 57, "hall": HALL},
        # The warm start's forward pass on both hemispheres at full grid.
        {"name": "unet_forward", "kind": "unet", "do": "forward", "h": 128, "w": 256, "batch": 2},
        # Loss and gradients of a training batch on the pooled polar grid.
        {"name": "unet_gradients_pooled", "kind": "unet", "do": "gradients", "h": 32, "w": 64,
         "batch": 8},
        # Loss and gradients of a training batch at full grid.
        {"name": "unet_gradients_full", "kind": "unet", "do": "gradients", "h": 128, "w": 256,
         "batch": 8},
        # Training steps on generated pairs of config1's polar grids, the
        # network on the grid pooled 4 x 4.
        {"name": "unet_train_pooled", "kind": "unet", "do": "train", "h": 32, "w": 64, "batch": 8,
         "pool": 4, "steps": 20},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "polar", "unet"])
    if kind == "step":
        nr, n = _log_int(rng, 8, 160), _log_int(rng, 10, 80)
        coupled = rng.random() < 0.3
        if coupled:
            # the innermost ghost cell stays above the ionosphere
            nr = max(nr, 16)
        return {"kind": "step", "nr": nr, "n": n, "steps": rng.choice([10, 20, 40]),
                "mixed": rng.random() < 0.3, "fidelity": rng.random() < 0.5,
                "graph": rng.random() < 0.5,
                "nt": _log_int(rng, 12, 64) if coupled else 0,
                "np": _log_int(rng, 32, 128) if coupled else 0,
                "hall": rng.choice([0.0, HALL]) if coupled else 0.0}
    if kind == "polar":
        return {"kind": "polar", "nt": _log_int(rng, 12, 140), "np": _log_int(rng, 24, 280),
                "hall": rng.choice([0.0, HALL])}
    do = rng.choice(["forward", "gradients"])
    return {"kind": "unet", "do": do, "h": 8 * rng.randint(2, 15), "w": 8 * rng.randint(4, 31),
            "batch": rng.randint(1, 8)}


# ---- inputs ------------------------------------------------------------------------------


def _earth(case, seed):
    wind = _ws.wind_variation(seed)
    kw = {}
    if case["nt"]:
        kw = dict(mi=True, hall_siemens=case["hall"], pedersen_siemens=PEDERSEN,
                  mi_azimuth=case["np"], mi_colatitude=case["nt"])
    return _cfg.earth_problem(case["nr"], case["n"], perturbation=0.01, seed=seed, **wind, **kw)


def _currents(nt, np_, seed):
    """Field-aligned current of two successive ionosphere updates
    ([2][nt][np] each, A/m^2): a region-1 / region-2 pair of sheets with
    smaller patches, of which the second update changes about a third."""
    rng = np.random.default_rng(seed)
    th = np.linspace(0.0, 1.0, nt)[:, None]
    ph = 2.0 * np.pi * np.arange(np_)[None, :] / np_

    def pattern():
        out = np.zeros((2, nt, np_))
        for h in range(2):
            turn = rng.uniform(0.0, 2.0 * np.pi)
            c1 = rng.uniform(0.45, 0.6)
            sheet = np.exp(-((th - c1) / 0.08) ** 2) - 0.6 * np.exp(-((th - c1 - 0.2) / 0.08) ** 2)
            out[h] = sheet * np.sin(ph - turn)
            for _ in range(6):
                d = (th - rng.uniform(0.1, 0.9)) / rng.uniform(0.04, 0.2)
                k = rng.uniform(0.5, 8.0)
                out[h] += 0.3 * rng.standard_normal() * np.exp(
                    -0.5 * d * d + k * (np.cos(ph - rng.uniform(0.0, 2.0 * np.pi)) - 1.0))
        out[:, 0] = out[:, -1] = 0.0
        return 1e-6 * out

    first = pattern()
    return first, first + 0.3 * pattern()


def _solve(current, hall):
    """The polar system's potential, [2][nt][np], in 64 bits: conductances
    are uniform, so a Fourier transform in longitude leaves one tridiagonal
    system in colatitude per wave number, solved densely. The pole is the
    mean of the first ring, the outer ring zero."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    fac = torch.from_numpy(current).to(dev)
    _, nt, np_ = fac.shape
    radius = 1.0 * _cfg.LENGTH_NORM_M
    dt = math.asin(math.sqrt(1.0 / 2.5)) / (nt - 1)
    dp = 2.0 * math.pi / np_
    i = torch.arange(1, nt - 1, dtype=torch.float64, device=dev)
    th = i * dt

    def cos_incl(t):
        return 2.0 * torch.cos(t) / torch.sqrt(1.0 + 3.0 * torch.cos(t) ** 2)

    def coupling(t):
        return torch.sin(t) * PEDERSEN / (cos_incl(t) ** 2 * dt * dt)

    lo, hi = coupling(th - 0.5 * dt), coupling(th + 0.5 * dt)
    lon = PEDERSEN / (torch.sin(th) * dp * dp)
    m = torch.arange(np_, dtype=torch.float64, device=dev)[:, None]
    out = torch.zeros_like(fac)
    for h, sign in ((0, -1.0), (1, 1.0)):
        drift = sign * hall * (1.0 / cos_incl(th - dt) - 1.0 / cos_incl(th + dt)) / (2.0 * dt)
        diag = (lo + hi + 2.0 * lon * (1.0 - torch.cos(m * dp))).to(torch.complex128)
        diag = diag - 1j * drift * torch.sin(m * dp) / dp
        diag[0, 0] -= lo[0]
        a = torch.diag_embed(diag)
        a = a + torch.diag_embed((-hi[:-1]).to(a.dtype), 1) + torch.diag_embed(
            (-lo[1:]).to(a.dtype), -1)
        rhs = -radius * radius * fac[h, 1:-1] * (sign * cos_incl(th) * torch.sin(th))[:, None]
        modes = torch.fft.fft(rhs, dim=1).T.contiguous()
        x = torch.linalg.solve(a, modes.unsqueeze(-1)).squeeze(-1)
        out[h, 1:-1] = torch.fft.ifft(x.T.contiguous(), dim=1).real
        out[h, 0] = out[h, 1].mean()
    return out.cpu().numpy()


def _net_inputs(case, seed):
    """Parameters (He-normal weights, small biases and head), features and
    targets of a batch."""
    rng = np.random.default_rng(seed)
    parts = []
    for cin, cout in LAYERS:
        parts.append(rng.standard_normal(cout * 9 * cin) * math.sqrt(2.0 / (9 * cin)))
        parts.append(0.05 * rng.standard_normal(cout))
    parts.append(0.2 * rng.standard_normal(32))
    parts.append(np.zeros(1))
    params = np.concatenate(parts).astype(np.float32)
    b, h, w = case["batch"], case["h"], case["w"]
    x = np.zeros((b, h, w, 32), dtype=np.float32)
    x[..., :16] = rng.standard_normal((b, h, w, 16), dtype=np.float32)
    x[..., 16] = rng.uniform(0.5, 1.5, (b, 1, 1))
    x[..., 17] = rng.uniform(0.0, 1.0, (b, 1, 1))
    x[..., 18] = np.linspace(0.0, 1.0, h)[None, :, None]
    x[..., 19] = rng.choice([-1.0, 1.0], (b, 1, 1))
    target = rng.standard_normal((b, h, w), dtype=np.float32)
    return params, x, target


def prepare(case, seed):
    if case["kind"] == "step":
        p = _native.GpuProblem(_earth(case, seed))
        p.set_fidelity(case["fidelity"])
        p.set_graph(case["graph"])
        if case["mixed"]:
            p.set_precision(True)
        # past the first steps, which recover every cell and make the first
        # ionosphere update
        p.advance(4)
        return {"case": case, "problem": p}
    if case["kind"] == "polar":
        p = _native.GpuProblem(_cfg.earth_problem(
            16, 12, perturbation=0.01, seed=7, mi=True, hall_siemens=case["hall"],
            pedersen_siemens=PEDERSEN, mi_azimuth=case["np"], mi_colatitude=case["nt"]))
        last, current = _currents(case["nt"], case["np"], seed)
        return {"case": case, "problem": p, "current": current,
                "guess": _solve(last, case["hall"])}
    net = _ws.WarmStartNet(case["h"], case["w"], case["batch"], seed=0)
    params, x, target = _net_inputs(case, seed)
    net.set_params(params)
    state = {"case": case, "net": net, "x": x, "target": target, "seed": seed}
    if case["do"] == "train":
        f = case["pool"]
        state["problem"] = _native.GpuProblem(_cfg.earth_problem(
            16, 12, perturbation=0.01, seed=7, mi=True, hall_siemens=HALL,
            pedersen_siemens=PEDERSEN, mi_azimuth=f * case["w"], mi_colatitude=f * case["h"]))
    return state


# ---- passes ------------------------------------------------------------------------------


class _View:
    """A view of an array that its problem owns, keeping the problem."""

    def __init__(self, array, owner):
        self.__array_interface__ = array.__array_interface__
        self.owner = owner


def _state(p):
    """Clock, conserved state, cell B and face fluxes of the active cells and
    faces (ghost values are storage, kept only on request)."""
    g, nr, n = p.config.ghost, p.config.radial_cells, p.config.angular_cells
    ni, nj, nk = p.config.extent
    c = p.clock()
    out = {"clock": np.array([c["time"], c["dt"], c["previous_dt"]])}
    box = (slice(g, g + nr), slice(g, g + n), slice(g, g + n))
    for f in range(_cfg.FACE_COUNT):
        for name, fid, nc in (("U", _problem.CONSERVED, 5), ("B", _problem.CELL_MAGNETIC, 3)):
            a = np.asarray(_View(p.field(f, fid), p))
            out[f"{name}{f}"] = a.reshape(ni, nj, nk, nc)[box]
        for d in range(3):
            ext = [ni, nj, nk]
            ext[d] += 1
            at = list(box)
            at[d] = slice(at[d].start, at[d].stop + 1)
            a = np.asarray(_View(p.field(f, _problem.FACE_FLUX + d), p))
            out[f"flux{f}{d}"] = a.reshape(ext)[tuple(at)]
    return out


def run(state):
    case = state["case"]
    if case["kind"] == "step":
        state["problem"].advance(case["steps"])
        return _state(state["problem"])
    if case["kind"] == "polar":
        potential, _, _ = _ws.solve_current(state["problem"], state["current"], state["guess"],
                                            use_network=False)
        return potential
    net = state["net"]
    if case["do"] == "forward":
        return net.forward(state["x"])
    if case["do"] == "gradients":
        loss = net.gradients(state["x"], state["target"])
        return {"loss": loss, "grads": net.grads()}
    losses = _ws.train(state["problem"], net, steps=case["steps"], batch=case["batch"],
                       seed=state["seed"])
    return {"losses": losses, "params": net.params()}


# ---- what a pass cannot do without ------------------------------------------------------


def _net_work(case):
    """(flops of one forward pass, parameters)."""
    b, h, w = case["batch"], case["h"], case["w"]
    flops, params = 0, 33
    for (cin, cout), lv in zip(LAYERS, LEVEL):
        flops += 2 * 9 * cin * cout * b * (h >> lv) * (w >> lv)
        params += cout * (9 * cin + 1)
    return flops + 64 * b * h * w, params


def work(case):
    if case["kind"] == "step":
        cells = 6 * case["nr"] * case["n"] ** 2
        return {"bytes": float(cells * (case["steps"] * STEP_BYTES + 2 * 11 * 8)),
                "flops": float(cells * case["steps"] * STEP_FLOPS)}
    if case["kind"] == "polar":
        # current and guess in, potential out; transforms in longitude and a
        # complex tridiagonal solve per wave number, one way to solve it
        n = 2 * case["nt"] * case["np"]
        return {"bytes": float(3 * 8 * n), "flops": float(n * (10 * math.log2(case["np"]) + 30))}
    pix = case["batch"] * case["h"] * case["w"]
    flops, params = _net_work(case)
    if case["do"] == "forward":
        return {"bytes": float(4 * (33 * pix + params)), "flops": float(flops)}
    if case["do"] == "gradients":
        return {"bytes": float(4 * (34 * pix + 2 * params)), "flops": float(3 * flops)}
    # per step: features and targets from the fine grid's pairs, parameters
    # and both moments read and written
    per = 4 * (34 * pix + 7 * params)
    return {"bytes": float(case["steps"] * per), "flops": float(case["steps"] * 3 * flops)}


def tolerance(case):
    # About four times what was seen, over one to three passes.
    if case["kind"] == "step":
        if case["mixed"]:
            # FP32 products fused or not in the sums: 8.7e-7, 7.8e-6
            return {"rel": 5e-6, "max": 5e-5}
        if case["nt"]:
            # the potential to 1e-10 or to 1e-12 of its right-hand side:
            # 2.6e-12, 2.8e-11
            return {"rel": 1e-11, "max": 1.2e-10}
        # FP64 products fused or not in the sums: 6.3e-15, 1.4e-13
        return {"rel": 3e-14, "max": 6e-13}
    if case["kind"] == "polar":
        # the solve stops at a residual of 1e-10 of the right-hand side:
        # 1.3e-10, 3e-10 from the exact potential
        return {"rel": 1e-9, "max": 5e-9}
    # bf16 activations and operands; against 64 bits: 8e-3, 3e-2 forward,
    # 1.1e-2, 0.2 (a single small sample: 2.2e-2, 0.5) in the gradients
    if case["do"] == "forward":
        return {"rel": 1e-2, "max": 1e-1}
    if case["do"] == "gradients":
        return {"rel": 2e-2, "max": 5e-1}
    # 20 Adam steps with fp32 sums in another order: 2.1e-3, 4.1e-2
    return {"rel": 1e-2, "max": 2e-1}


# ---- the same in 64 bits ------------------------------------------------------------------


def _conv(x, w, b):
    """3x3 convolution, NHWC, zero rows beyond the first axis' ends and
    periodic columns; w [cout][3][3][cin]."""
    wide = torch.cat([x[:, :, -1:], x, x[:, :, :1]], dim=2)
    zero = torch.zeros_like(wide[:, :1])
    wide = torch.cat([zero, wide, zero], dim=1)
    h, wd = x.shape[1], x.shape[2]
    out = b
    for ky in range(3):
        for kx in range(3):
            out = out + wide[:, ky:ky + h, kx:kx + wd].reshape(-1, x.shape[3]).matmul(
                w[:, ky, kx].t().contiguous()).reshape(x.shape[0], h, wd, -1)
    return torch.relu(out)


def _forward64(params, x):
    layers, at = [], 0
    for cin, cout in LAYERS:
        w = params[at:at + cout * 9 * cin].reshape(cout, 3, 3, cin)
        at += cout * 9 * cin
        layers.append((w, params[at:at + cout]))
        at += cout
    head, bias = params[at:at + 32], params[at + 32]

    def block(k, v):
        return _conv(_conv(v, *layers[k]), *layers[k + 1])

    def pool(v):
        n, h, w, c = v.shape
        return v.reshape(n, h // 2, 2, w // 2, 2, c).mean(dim=(2, 4))

    def up(v):
        return v.repeat_interleave(2, dim=1).repeat_interleave(2, dim=2)

    e0 = block(0, x)
    e1 = block(2, pool(e0))
    e2 = block(4, pool(e1))
    e3 = block(6, pool(e2))
    d2 = block(8, torch.cat([up(e3), e2], dim=3))
    d1 = block(10, torch.cat([up(d2), e1], dim=3))
    d0 = block(12, torch.cat([up(d1), e0], dim=3))
    return d0.matmul(head) + bias


def exact(case, seed):
    if case["kind"] == "step":
        # tens of MHD steps of a few thousand operations a cell; there is no
        # short plain form of them
        return None
    if case["kind"] == "polar":
        return _solve(_currents(case["nt"], case["np"], seed)[1], case["hall"])
    if case["do"] == "train":
        # the pairs come from the library's own generator
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    params, x, target = _net_inputs(case, seed)
    p = torch.from_numpy(params).double().to(dev).requires_grad_(case["do"] == "gradients")
    out = _forward64(p, torch.from_numpy(x).double().to(dev))
    if case["do"] == "forward":
        return out.detach()
    loss = (out - torch.from_numpy(target).double().to(dev)).square().mean()
    loss.backward()
    return {"loss": loss.item(), "grads": p.grad}

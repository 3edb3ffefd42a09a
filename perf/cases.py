"""The work that programs using this framework have it do, as timed cases.

Each case is one call of a program's main path: a time step of a solver, a
step of an ensemble, a transform, a set of outputs, a training step of the
closure network.  ``listed`` gives the named ones, ``draw`` further ones of
the same ranges.  ``prepare`` builds what the program holds before the call
(from the seed alone), ``run`` makes the call, ``exact`` restates its result
in 64 bits with plain torch.
"""

import contextlib
import io
import os
import random
import tempfile
from math import log2, pi

import numpy as np
import torch

PHASESHIFT_COEF = 2.0 * 2**0.5 / 3  # truncation radius of the phase-shifted schemes

# transforms per evaluation of the nonlinear term, state variables
TRANSFORMS = {"ns2d": 5, "ns3d": 9, "ns3d.strat": 13}
NVAR = {"ns2d": 1, "ns3d": 3, "ns3d.strat": 4}
STAGES = {"RK4": 4, "RK2": 2, "RK2_phaseshift": 2}


def _step(solver, shape, precision, scheme="RK4", truncation="cubic", forced=False):
    return {"kind": "step", "solver": solver, "nx": shape[0], "ny": shape[1],
            "nz": shape[2] if len(shape) > 2 else 1, "precision": precision,
            "scheme": scheme, "truncation": truncation, "forced": forced}


def _named(name, case):
    return {"name": name, **case}


def listed():
    return [
        # the solvers' default grid, a length that is not a power of two: a
        # first script, a parameter scan, a test; all latency
        _named("ns2d_48_f64", _step("ns2d", (48, 48), "float64")),
        # the usual small 2D run, adaptive dt, in the default precision
        _named("ns2d_256_f64", _step("ns2d", (256, 256), "float64")),
        # forced 2D turbulence at the resolution of the closure's DNS
        _named("ns2d_2048_f32_forced", _step("ns2d", (2048, 2048), "float32", forced=True)),
        # many independent 2D runs of three sizes, one graph launch per step
        _named("ensemble_512_runs", {"kind": "ensemble", "n0": 128, "count0": 256, "n1": 256,
                                     "count1": 192, "n2": 512, "count2": 64}),
        # 3D turbulence production run, FP32
        _named("ns3d_512_f32", _step("ns3d", (512, 512, 512), "float32")),
        # the recommended anti-aliasing set-up: phase-shifted RK2 with the
        # truncation that keeps more modes (not a box), double precision
        _named("ns3d_256_f64_phaseshift",
               _step("ns3d", (256, 256, 256), "float64", "RK2_phaseshift",
                     "no_multiple_aliases")),
        # stratified turbulence in a flat box, long horizontal axes
        _named("strat_1024_1024_256_f32", _step("ns3d.strat", (1024, 1024, 256), "float32")),
        # 3D grid of ragged lengths (5-smooth), as FFT libraries allow
        _named("ns3d_240_192_160_f64", _step("ns3d", (240, 192, 160), "float64")),
        # the operators alone: a vector field to spectral space and back,
        # what scripts and post-processing call
        _named("transform_512_f32", {"kind": "transform", "nx": 512, "ny": 512, "nz": 512,
                                     "fields": 3, "precision": "float32"}),
        # the periodic outputs of a 3D run: all spectra and the means
        _named("outputs_512_f32", {"kind": "outputs", "nx": 512, "ny": 512, "nz": 512,
                                   "precision": "float32"}),
        # one Adam step of the closure network on a batch of 2D fields
        _named("train_32x128", {"kind": "train", "batch": 32, "n": 128}),
        # LES with the learned term in every stage, on its usual coarse grid
        _named("les_128_f32", {"kind": "les", "n": 128, "precision": "float32"}),
    ]


def _ragged(rng, lo, hi):
    """A length in [lo, hi], spread over its logarithm: a power of two, an
    even or odd product of small primes, or any integer with prime factors
    up to 31."""
    how = rng.random()
    target = lo * (hi / lo) ** rng.random()
    if how < 0.4:
        return min(hi, max(lo, 2 ** round(log2(target))))
    limit = 7 if how < 0.85 else 31
    n = int(target)
    while True:
        m = n
        for p in (2, 3, 5, 7, 11, 13, 17, 19, 23, 29, 31):
            while p <= limit and m % p == 0:
                m //= p
        if m == 1:
            return n
        n += 1 if n < hi else -1


def draw(rng):
    kind = rng.choices(["ns2d", "ns3d", "ns3d.strat", "ensemble", "transform", "outputs",
                        "train", "les"], [4, 4, 3, 2, 2, 2, 2, 1])[0]
    precision = rng.choice(["float32", "float64"])
    if kind == "ns2d":
        hi = 2048 if precision == "float32" else 1024
        return _step("ns2d", (_ragged(rng, 32, hi), _ragged(rng, 32, hi)), precision,
                     rng.choice(["RK4", "RK4", "RK2", "RK2_phaseshift"]), "cubic",
                     rng.random() < 0.3)
    if kind in ("ns3d", "ns3d.strat"):
        hi = 512 if precision == "float32" else 256
        shape = [_ragged(rng, 24, hi) for _ in range(3)]
        ragged = any(n & (n - 1) for n in shape)
        while shape[0] * shape[1] * shape[2] > (2**23 if ragged else 2**26):
            i = shape.index(max(shape))
            shape[i] = _ragged(rng, 24, shape[i])
        scheme, truncation = rng.choice([("RK4", "cubic"), ("RK4", "spherical"),
                                         ("RK2", "cubic"),
                                         ("RK2_phaseshift", "no_multiple_aliases")])
        return _step(kind, shape, precision, scheme, truncation)
    if kind == "ensemble":
        sizes = rng.sample([32, 64, 128, 256, 512], 3)
        case = {"kind": "ensemble"}
        for i, n in enumerate(sorted(sizes)):
            case[f"n{i}"] = n
            case[f"count{i}"] = rng.randint(1, min(300, 64 * 512**2 // n**2))
        return case
    if kind in ("transform", "outputs"):
        shape = [_ragged(rng, 24, 512) for _ in range(3)]
        while shape[0] * shape[1] * shape[2] > 2**25:
            i = shape.index(max(shape))
            shape[i] = _ragged(rng, 24, shape[i])
        case = {"kind": kind, "nx": shape[0], "ny": shape[1], "nz": shape[2],
                "precision": precision}
        if kind == "transform":
            case["fields"] = rng.randint(1, 3)
        return case
    if kind == "train":
        n = rng.choice([32, 64, 96, 128])
        return {"kind": "train", "batch": rng.randint(2, 32 * 128**2 // max(n, 128) ** 2),
                "n": n}
    return {"kind": "les", "n": rng.choice([32, 64, 96, 128, 160, 192, 256]),
            "precision": "float32"}


# ------------------------------------------------------------------ inputs
def _complex(precision):
    return torch.complex64 if precision == "float32" else torch.complex128


def _lengths(case):
    """Box of an isotropic mesh, the longest side 2 pi."""
    ns = [case["nx"], case["ny"]] + ([case["nz"]] if case["nz"] > 1 else [])
    return [2 * pi * n / max(ns) for n in ns]


class _Grid:
    """64-bit wavenumbers, masks and transforms of a case's grid (arrays in
    the order z, y, x), in plain torch."""

    def __init__(self, ns, lengths, truncation="cubic", coef=2.0 / 3):
        self.ns, self.lengths = ns, lengths
        self.nx = ns[0]
        self.shape = tuple(reversed(ns))
        self.shapeK = self.shape[:-1] + (ns[0] // 2 + 1,)
        self.axes = tuple(range(-len(ns), 0))
        self.deltas = [L / n for L, n in zip(lengths, ns)]
        self.dk = [2 * pi / L for L in lengths]
        self.k = []  # x, y(, z), broadcastable
        for axis, (n, dk) in enumerate(zip(ns, self.dk)):
            i = torch.arange(n // 2 + 1 if axis == 0 else n, dtype=torch.float64, device="cuda")
            if axis > 0:
                i = torch.where(i <= n // 2, i, i - n)
            shape = [1] * len(ns)
            shape[len(ns) - 1 - axis] = len(i)
            self.k.append((dk * i).reshape(shape))
        self.k2 = sum(k * k for k in self.k)
        self.k2_not0 = torch.where(self.k2 == 0, 1e-14, self.k2)
        cut = [k.abs() >= coef * dk * n / 2 for k, dk, n in zip(self.k, self.dk, ns)]
        kmax2 = (coef * self.dk[0] * ns[0] / 2) ** 2
        if truncation == "cubic":
            out = cut[0]
            for c in cut[1:]:
                out = out | c
        elif truncation == "spherical":
            out = self.k2 >= kmax2
        else:
            a = [k.abs() >= 2 / 3 * dk * n / 2 for k, dk, n in zip(self.k, self.dk, ns)]
            if len(a) == 2:
                out = (a[0] & a[1]) | (self.k2 >= kmax2)
            else:
                out = ((a[0] & a[1]) | (a[1] & a[2]) | (a[2] & a[0])) | (self.k2 >= kmax2)
        self.keep = ~out

    def fft(self, x):
        return torch.fft.rfftn(x, dim=self.axes, norm="forward")

    def ifft(self, a):
        return torch.fft.irfftn(a, s=self.shape, dim=self.axes, norm="forward")

    def weights(self):
        w = torch.full((self.nx // 2 + 1,), 2.0, dtype=torch.float64, device="cuda")
        w[0] = 1.0
        if self.nx % 2 == 0:
            w[-1] = 1.0
        return w


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _random_field(grid, g, amplitude, lead=()):
    x = torch.randn(tuple(lead) + grid.shape, generator=g, device="cuda", dtype=torch.float64)
    return grid.fft(x) * (amplitude * grid.keep)


def _vorticity(grid, g, lead=()):
    """Band-limited turbulent vorticity: energy around mode 8 with a k^-3
    tail, largest velocity about 1."""
    k = grid.k2_not0.sqrt()
    k0 = min(8.0, max(grid.ns) / 8) * min(grid.dk)
    rot = _random_field(grid, g, k**2 / (k0 + k) ** 3.5 * (grid.k2 > 0), lead)
    speed2 = sum(grid.ifft(1j * q * rot / grid.k2_not0) ** 2 for q in grid.k)
    return rot / speed2.amax(dim=grid.axes, keepdim=True).sqrt()


def _velocity(grid, g, nvar):
    """Solenoidal turbulent velocity (energy around mode 4, k^-5/3 tail, unit
    energy); the fourth variable (buoyancy) with the same spectrum."""
    k = grid.k2_not0.sqrt()
    k0 = min(4.0, max(grid.ns) / 8) * min(grid.dk)
    amp = k / (k0 + k) ** (17 / 6) * (grid.k2 > 0)
    v = [_random_field(grid, g, amp) for _ in range(nvar)]
    div = sum(k * a for k, a in zip(grid.k, v)) / grid.k2_not0
    for i in range(3):
        v[i] -= grid.k[i] * div
    w = grid.weights()
    energy = sum(float((w * (a.real**2 + a.imag**2)).sum()) for a in v[:3]) / 2
    return torch.stack(v) / energy**0.5


def _step_grid(case):
    ns = [case["nx"], case["ny"]] + ([case["nz"]] if case["nz"] > 1 else [])
    coef = PHASESHIFT_COEF if case["truncation"] == "no_multiple_aliases" else 2.0 / 3
    return _Grid(ns, _lengths(case), case["truncation"], coef), coef


def _step_state(case, seed, grid):
    g = _generator(seed)
    if case["solver"] == "ns2d":
        state = _vorticity(grid, g)[None]
    else:
        state = _velocity(grid, g, NVAR[case["solver"]])
    return state.to(_complex(case["precision"]))


def _viscosity(case, grid):
    """nu_2 of the 2D runs, nu_8 of the 3D ones (largest kept wavenumber
    about dissipative)."""
    kmax = 2 / 3 * grid.dk[0] * grid.ns[0] / 2
    if case["solver"] == "ns2d":
        return {"nu_2": 0.5 / kmax**2}
    return {"nu_8": kmax ** (-22.0 / 3.0)}


BRUNT_VAISALA = 4.0
NKMIN, NKMAX = 8, 10  # forced shells of the forced runs


def _nk(n):
    """Forced shells of an n-point axis: 8 to 10, fewer on short axes."""
    return (NKMIN, NKMAX) if n >= 64 else (2, 3)


def _simul(Simul, params, case, coef, lengths):
    params.oper.nx, params.oper.ny = case["nx"], case["ny"]
    params.oper.Lx, params.oper.Ly = lengths[0], lengths[1]
    if case["nz"] > 1:
        params.oper.nz, params.oper.Lz = case["nz"], lengths[2]
    params.oper.precision = case["precision"]
    params.oper.coef_dealiasing = coef
    params.oper.truncation_shape = case["truncation"]
    params.time_stepping.type_time_scheme = case["scheme"]
    params.time_stepping.USE_CFL = True
    params.time_stepping.cfl_coef = 0.5
    params.init_fields.type = "in_script"
    params.output.HAS_TO_SAVE = False
    params.output.periods_print.print_stdout = 0
    if case["forced"]:
        params.forcing.enable = True
        params.forcing.type = "tcrandom"
        params.forcing.nkmin_forcing, params.forcing.nkmax_forcing = _nk(
            min(case["nx"], case["ny"]))
        params.forcing.forcing_rate = 1.0
    with contextlib.redirect_stdout(io.StringIO()):
        return Simul(params)


def _set_state(sim, state):
    sim.state.init_statespect_from(**dict(zip(sim.state.keys_state_spect, state)))


def _prepare_step(case, seed):
    from importlib import import_module

    Simul = import_module(f"fluidsim_amd.solvers.{case['solver']}.solver").Simul
    grid, coef = _step_grid(case)
    params = Simul.create_default_params()
    for key, value in _viscosity(case, grid).items():
        setattr(params, key, value)
    if case["solver"] == "ns3d.strat":
        params.N = BRUNT_VAISALA
    np.random.seed(seed % 2**31)
    sim = _simul(Simul, params, case, coef, _lengths(case))
    _set_state(sim, _step_state(case, seed, grid))
    sim.time_stepping.prepare_main_loop()
    return sim


def _runs(case):
    return [(case[f"n{i}"], case[f"count{i}"]) for i in range(3)]


def _ensemble_inputs(case, seed):
    """Per size: vorticities (count, n, n/2 + 1) and viscosities."""
    g = _generator(seed)
    rng = random.Random(seed)
    out = []
    for n, count in _runs(case):
        grid = _Grid([n, n], [2 * pi, 2 * pi])
        rot = torch.cat([_vorticity(grid, g, (min(32, count - i),)).to(torch.complex64)
                         for i in range(0, count, 32)])
        out.append((grid, rot, [10 ** rng.uniform(-4, -2) for _ in range(count)]))
    return out


def _prepare_ensemble(case, seed):
    from fluidsim_amd.ensemble import EnsembleNS2D

    runs = []
    for grid, rot, nus in _ensemble_inputs(case, seed):
        rot = rot.cpu().numpy()
        runs += [{"n": grid.nx, "rot_fft": r, "nu_2": nu} for r, nu in zip(rot, nus)]
    # a tuning table of this process, as after a first run of the program
    cache = os.path.join(tempfile.gettempdir(), f"ensemble_tuning_{os.getpid()}.json")
    return EnsembleNS2D(runs, precision="float32", tune_cache=cache)


def _transform_input(case, seed):
    grid = _Grid([case["nx"], case["ny"], case["nz"]], _lengths(case))
    g = _generator(seed)
    real = torch.float32 if case["precision"] == "float32" else torch.float64
    return torch.randn((case["fields"],) + grid.shape, generator=g, device="cuda", dtype=real)


def _prepare_transform(case, seed):
    from fluidsim_amd.operators.operators3d import OperatorsPseudoSpectral3D as Operators

    params = Operators._create_default_params()
    lengths = _lengths(case)
    params.oper.nx, params.oper.ny, params.oper.nz = case["nx"], case["ny"], case["nz"]
    params.oper.Lx, params.oper.Ly, params.oper.Lz = lengths
    params.oper.precision = case["precision"]
    return Operators(params), _transform_input(case, seed)


def _outputs_step(case):
    return _step("ns3d", (case["nx"], case["ny"], case["nz"]), case["precision"])


def _closure_net(seed):
    """A network with non-zero biases, as after some training."""
    from fluidsim_amd.closure import CNNClosure

    net = CNNClosure(n_in=1, nlayers=6, seed=seed % 2**31)
    rng = np.random.default_rng(seed + 1)
    weights = net.state_dict()
    for layer, (_, co) in enumerate(_layers()):
        weights[f"b{layer}"][:co] = 0.05 * rng.standard_normal(co)
    net.load_state_dict(weights)
    return net


def _train_batch(case, seed):
    """Normalised vorticity and subgrid term: smooth random fields of unit
    variance, the target nearly a local function of the input."""
    grid = _Grid([case["n"], case["n"]], [2 * pi, 2 * pi])
    rot = grid.ifft(_vorticity(grid, _generator(seed), (case["batch"],)))
    x = rot / rot.std()
    y = torch.tanh(x) * torch.roll(x, (1, 2), (1, 2))
    return x[..., None].float().contiguous(), (y / y.std()).float().contiguous()


def _prepare_train(case, seed):
    return (_closure_net(seed),) + _train_batch(case, seed)


LES_IN, LES_OUT = 8.0, 0.5  # scales of the vorticity and of the learned term


def _les_step(case):
    return _step("ns2d", (case["n"], case["n"]), case["precision"], forced=True)


def _prepare_les(case, seed):
    from fluidsim_amd.closure import make_les_class

    step = _les_step(case)
    grid, coef = _step_grid(step)
    Simul = make_les_class()
    params = Simul.create_default_params()
    params.nu_2 = _viscosity(step, grid)["nu_2"]
    np.random.seed(seed % 2**31)
    sim = _simul(Simul, params, step, coef, _lengths(step))
    _set_state(sim, _step_state(step, seed, grid))
    sim.closure_net = _closure_net(seed).folded(LES_IN, LES_OUT)
    sim.time_stepping.prepare_main_loop()
    return sim


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        state = _prepare_step(case, seed)
    elif kind == "ensemble":
        state = _prepare_ensemble(case, seed)
    elif kind == "transform":
        state = _prepare_transform(case, seed)
    elif kind == "outputs":
        state = _prepare_step(_outputs_step(case), seed)
    elif kind == "train":
        state = _prepare_train(case, seed)
    else:
        state = _prepare_les(case, seed)
    return {"kind": kind, "state": state}


# ------------------------------------------------------------------ the call
def run(state):
    kind, s = state["kind"], state["state"]
    if kind in ("step", "les"):
        s.time_stepping.one_time_step()
        return s.state.state_spect.data, float(s.time_stepping.deltat)
    if kind == "ensemble":
        # the ensemble works on a stream of its own
        cur = torch.cuda.current_stream()
        s.stream.wait_stream(cur)
        s.step()
        cur.wait_stream(s.stream)
        return [g.S for g in s.groups]
    if kind == "transform":
        oper, x = s
        x_fft = oper.fft3d(x)
        return x_fft, oper.ifft3d(x_fft)
    if kind == "outputs":
        spectra = s.output.spectra.compute(kzkh=True)
        return list(spectra) + [s.output.spatial_means.compute()]
    net, x, y = s
    net.train_step(x, y, want_loss=False)
    return list(net.last_grads[0]), list(net.last_grads[1]), list(net.w), list(net.b)


# ------------------------------------------------------------------ its cost
def _fft_flops(shape):
    n = 1
    for m in shape:
        n *= m
    return 2.5 * n * log2(n)


def _layers():
    """Channels in and out of the network's six layers."""
    return [(1, 32)] + [(32, 32)] * 4 + [(32, 1)]


def work(case):
    kind = case["kind"]
    if kind == "step":
        csize = 8 if case["precision"] == "float32" else 16
        shape = (case["nx"], case["ny"], case["nz"])
        modes = (case["nx"] // 2 + 1) * case["ny"] * case["nz"]
        nvar, stages = NVAR[case["solver"]], STAGES[case["scheme"]]
        points = shape[0] * shape[1] * shape[2]
        return {"bytes": 2.0 * nvar * modes * csize,
                "flops": stages * (TRANSFORMS[case["solver"]] * _fft_flops(shape)
                                   + 5.0 * TRANSFORMS[case["solver"]] * points)}
    if kind == "ensemble":
        byts = flops = 0.0
        for n, count in _runs(case):
            one = work(_step("ns2d", (n, n), "float32"))
            byts += count * one["bytes"]
            flops += count * one["flops"]
        return {"bytes": byts, "flops": flops}
    if kind == "transform":
        size = 4 if case["precision"] == "float32" else 8
        points = case["nx"] * case["ny"] * case["nz"]
        modes = (case["nx"] // 2 + 1) * case["ny"] * case["nz"]
        return {"bytes": 2.0 * case["fields"] * size * (points + 2 * modes),
                "flops": 2.0 * case["fields"] * _fft_flops((points,))}
    if kind == "outputs":
        csize = 8 if case["precision"] == "float32" else 16
        modes = (case["nx"] // 2 + 1) * case["ny"] * case["nz"]
        return {"bytes": 2.0 * 3 * csize * modes, "flops": 100.0 * modes}
    if kind == "train":
        points = case["batch"] * case["n"] ** 2
        macs = sum(25 * a * b for a, b in _layers())
        first = 25 * 32
        weights = sum(32 * 25 * (8 if a == 1 else 32) for a, _ in _layers())
        return {"bytes": 8.0 * points + 28.0 * weights,
                "flops": 2.0 * points * (3 * macs - first)}
    step = work(_les_step(case))
    macs = sum(25 * a * b for a, b in _layers())
    return {"bytes": step["bytes"] + 2.0 * macs,
            "flops": step["flops"] + 4 * (2.0 * macs * case["n"] ** 2
                                          + 2 * _fft_flops((case["n"], case["n"])))}


def tolerance(case):
    if case["kind"] == "train":
        # BF16 activations and gradients: 1e-2 from 64 bits
        return {"rel": 2e-2}
    if case["kind"] == "les":
        return {"rel": 4e-6}
    if case["kind"] == "outputs":
        return {"rel": 1e-13}  # sums in 64 bits
    if case.get("precision", "float32") == "float64":
        return {"rel": 4e-15}
    return {"rel": 1e-6}


# ------------------------------------------------------------------ 64 bits
def _velocity_2d(grid, rot):
    return 1j * grid.k[1] * rot / grid.k2_not0, -1j * grid.k[0] * rot / grid.k2_not0


def _nonlinear(solver, grid, S):
    """Dealiased (and, in 3D, projected) nonlinear term of the state S."""
    if solver == "ns2d":
        rot = S[0]
        ux, uy = (grid.ifft(a) for a in _velocity_2d(grid, rot))
        gx, gy = (grid.ifft(1j * k * rot) for k in grid.k)
        return (grid.fft(-ux * gx - uy * gy) * grid.keep)[None]
    kx, ky, kz = grid.k
    v = [grid.ifft(a) for a in S[:3]]
    w = [grid.ifft(a) for a in (1j * (ky * S[2] - kz * S[1]), 1j * (kz * S[0] - kx * S[2]),
                                1j * (kx * S[1] - ky * S[0]))]
    N = torch.empty_like(S)
    N[0] = grid.fft(v[1] * w[2] - v[2] * w[1])
    N[1] = grid.fft(v[2] * w[0] - v[0] * w[2])
    N[2] = grid.fft(v[0] * w[1] - v[1] * w[0])
    del w
    if solver == "ns3d.strat":
        N[2] += S[3]
        b = grid.ifft(S[3])
        N[3] = -BRUNT_VAISALA**2 * S[2]
        for k, a in zip(grid.k, v):
            N[3] -= 1j * k * grid.fft(a * b)
    N *= grid.keep
    _project(grid, N)
    return N


def _project(grid, S):
    t = sum(k * a for k, a in zip(grid.k, S)) / grid.k2_not0
    for i in range(3):
        S[i] -= grid.k[i] * t


def _cfl_dt(solver, grid, S, cfl=0.5, dt_max=0.2):
    v = _velocity_2d(grid, S[0]) if solver == "ns2d" else S[:3]
    return min(cfl / sum(float(grid.ifft(a).abs().max()) / d
                         for a, d in zip(v, grid.deltas)), dt_max)


def _forcing(grid, seed, S, dt):
    """The normalised forcing (rate 1) of the first step of a forced 2D run:
    seeded random coarse modes in the forced ring."""
    nkmin, nkmax = _nk(min(grid.ns))
    nc = 1
    while nc < 2 * nkmax:
        nc *= 2
    i = np.arange(nc)
    ix, iy = np.arange(nc // 2 + 1), np.where(i <= nc // 2, i, i - nc)
    K = np.hypot(grid.dk[0] * ix[None, :], grid.dk[1] * iy[:, None])
    dk = max(grid.dk)
    ring = (K <= dk * nkmax) & (K >= dk * nkmin)
    ring[nc // 2, :] = False
    ring[:, nc // 2] = False
    np.random.seed(seed % 2**31)
    np.random.seed(np.random.randint(0, 2**31))
    re, im = np.random.random(ring.shape), np.random.random(ring.shape)
    f = np.where(ring, (2 * re - 1) + 1j * (2 * im - 1), 0)
    # Hermitian on the kx = 0 column: the spectrum of a real field
    f[:, 0] = (f[:, 0] + np.conj(f[-i % nc, 0])) / 2
    full = torch.zeros_like(S)
    rows = torch.from_numpy(np.where(iy < 0, iy + grid.ns[1], iy)).cuda()
    use = (iy > -nc // 2) & (iy <= nc // 2)
    full[0][rows[torch.from_numpy(use).cuda()], : nc // 2 + 1] = torch.from_numpy(f[use]).cuda()
    w = grid.weights()
    a = dt / 2 * float((w * full[0].abs() ** 2).sum())
    b = float((w * (S[0].conj() * full[0]).real).sum())
    root = (b * b + 4 * a) ** 0.5
    r1, r2 = (-b + root) / (2 * a), (-b - root) / (2 * a)
    return full * (r2 if abs(r2) < abs(r1) else r1)


def _advance(solver, grid, scheme, S, dt, visc, extra=None):
    """One step of the integrating-factor scheme; extra(S): further terms
    of the tendency."""
    sig = visc.get("nu_2", 0.0) * grid.k2 + visc.get("nu_8", 0.0) * grid.k2**4
    E, E2 = torch.exp(-dt * sig), torch.exp(-dt / 2 * sig)
    del sig

    def tend(x):
        N = _nonlinear(solver, grid, x)
        if extra is not None:
            N += extra(x)
        return N

    if scheme == "RK4":
        N = tend(S)
        tmp, t1 = (S + dt / 6 * N) * E, (S + dt / 2 * N) * E2
        N = tend(t1)
        tmp, t1 = tmp + dt / 3 * E2 * N, S * E2 + dt / 2 * N
        N = tend(t1)
        tmp, t1 = tmp + dt / 3 * E2 * N, S * E + dt * E2 * N
        return tmp + dt / 6 * tend(t1)
    if scheme == "RK2":
        return S * E + dt * E2 * tend((S + dt / 2 * tend(S)) * E2)
    # RK2_phaseshift: the second evaluation on a grid shifted by half a mesh
    phase = torch.exp(0.5j * sum(k * d for k, d in zip(grid.k, grid.deltas)))
    N0 = tend(S)
    N1 = tend((S + dt * N0) * E * phase) / phase
    return S * E + dt / 2 * E2 * (N0 + N1)


def _exact_step(case, seed, net=None):
    solver = case["solver"]
    grid, _ = _step_grid(case)
    S = _step_state(case, seed, grid).to(torch.complex128)
    dt = _cfl_dt(solver, grid, S)
    if abs(0.2 - dt) / dt <= 0.02:
        dt = 0.2  # within the hysteresis of the initial value
    extra = None
    if case["forced"] or net is not None:
        F = _forcing(grid, seed, S, dt) if case["forced"] else 0.0

        def extra(x):
            if net is None:
                return F
            y = _network(net, grid.ifft(x))
            return F + grid.fft(y) * grid.keep

    S = _advance(solver, grid, case["scheme"], S, dt, _viscosity(case, grid), extra)
    if solver != "ns2d":
        _project(grid, S)
    return S * grid.keep, dt


def _exact_ensemble(case, seed):
    out = []
    for grid, rot, nus in _ensemble_inputs(case, seed):
        parts = []
        for i, nu in enumerate(nus):
            S = rot[i].to(torch.complex128)[None]
            dt = _cfl_dt("ns2d", grid, S)
            parts.append(_advance("ns2d", grid, "RK4", S, dt, {"nu_2": nu}) * grid.keep)
        out.append(torch.cat(parts))
    return out


def _exact_outputs(case, seed):
    step = _outputs_step(case)
    grid, _ = _step_grid(step)
    S = _step_state(step, seed, grid).to(torch.complex128)
    kx, ky, kz = grid.k
    w = grid.weights()
    kh2 = kx**2 + ky**2
    kh2n = torch.where(kh2 == 0, 1e-14, kh2)
    fields = {c: 0.5 * (a.real**2 + a.imag**2) * w for c, a in zip(("vx", "vy", "vz"), S)}
    # rotational and divergent parts of the horizontal velocity
    rot, div = (kx * S[1] - ky * S[0]).abs() ** 2, (kx * S[0] + ky * S[1]).abs() ** 2
    fields["Khr"], fields["Khd"] = 0.5 * rot / kh2n * w, 0.5 * div / kh2n * w
    n = [grid.ns[i] // 2 + 1 for i in range(3)]
    dk, dkh = max(grid.dk), max(grid.dk[:2])
    nk = max(2, int(min(d * m for d, m in zip(grid.dk, n)) / dk))
    nkh = max(2, int(min(d * m for d, m in zip(grid.dk[:2], n[:2])) / dkh))

    def fold(axis):
        i = torch.arange(grid.ns[axis], device="cuda")
        return torch.where(i <= grid.ns[axis] // 2, i, grid.ns[axis] - i)

    def share(k, d, m):
        j = (k / d).long()
        last = j >= m - 1
        c = torch.where(last, 0.0, (k - j * d) / d)
        return torch.where(last, m - 1, j), c

    def histogram(q, j, c, size):
        h = torch.zeros(size + 1, dtype=torch.float64, device="cuda")
        h.index_add_(0, j.reshape(-1), ((1 - c) * q).reshape(-1))
        h.index_add_(0, (j + 1).reshape(-1), (c * q).reshape(-1))
        return h[:size]

    def line(q, axis, m, d):
        h = torch.zeros(m, dtype=torch.float64, device="cuda")
        return h.index_add_(0, fold(axis), q) / d

    j3, c3 = share(grid.k2.sqrt(), dk, nk)
    jh, ch = share(kh2.sqrt(), dkh, nkh)
    jz = fold(2)
    d1, d3, dh = {}, {}, {}
    for name, q in fields.items():
        d1[name + "_kx"] = q.sum((0, 1)) / grid.dk[0]
        d1[name + "_ky"] = line(q.sum((0, 2)), 1, n[1], grid.dk[1])
        d1[name + "_kz"] = line(q.sum((1, 2)), 2, n[2], grid.dk[2])
        d3[name] = histogram(q, j3, c3, nk) / dk
        planes = torch.stack([histogram(p, jh, ch, nkh) for p in q])
        z = torch.zeros((n[2], nkh), dtype=torch.float64, device="cuda")
        dh[name] = z.index_add_(0, jz, planes) / (grid.dk[2] * dkh)
    for ax in ("kx", "ky", "kz"):
        d1["E_" + ax] = d1["vx_" + ax] + d1["vy_" + ax] + d1["vz_" + ax]
    d3["E"] = d3["vx"] + d3["vy"] + d3["vz"]
    names = ("vx", "vy", "vz", "E", "Khr", "Khd")
    d1 = {f"{c}_{ax}": d1[f"{c}_{ax}"] for c in names for ax in ("kx", "ky", "kz")}
    d3 = {c: d3[c] for c in names}
    nu8 = _viscosity(step, grid)["nu_8"]
    energies = [float(fields[c].sum()) for c in ("vx", "vy", "vz")]
    eps = float((2 * nu8 * grid.k2**4 * (fields["vx"] + fields["vy"] + fields["vz"])).sum())
    means = {"E": sum(energies), "Ex": energies[0], "Ey": energies[1], "Ez": energies[2],
             "epsK": eps, "epsK_hypo": 0.0, "epsK_tot": eps, "epsK8": eps}
    host = [{"spectra_" + k: v.cpu().numpy() for k, v in d.items()} for d in (d1, d3)]
    kzkh = {"K": dh["vx"] + dh["vy"] + dh["vz"], "Khr": dh["Khr"], "Khd": dh["Khd"]}
    return host + [{k: v.cpu().numpy() for k, v in kzkh.items()}] + [means]


def _network_arrays(seed):
    """FP32 weights [co][ci][5][5] and biases of a network of this seed."""
    state = _closure_net(seed).state_dict()
    w, b = [], []
    for layer, (ci, co) in enumerate(_layers()):
        a = state[f"w{layer}"][:co, :, :ci].astype(np.float64)
        w.append(torch.from_numpy(a).cuda())
        b.append(torch.from_numpy(state[f"b{layer}"][:co].astype(np.float64)).cuda())
    return w, b


def _convolution(x, w, b):
    """Periodic 5x5 convolution of x (B, H, W, ci), weights (co, 25, ci)."""
    y = b
    for t in range(25):
        shifted = torch.roll(x, (2 - t // 5, 2 - t % 5), (1, 2))
        y = y + (shifted.reshape(-1, x.shape[-1]) @ w[:, t].T).reshape(*x.shape[:3], -1)
    return y


def _network(net, x):
    """Network (weights, biases) on fields x (B, H, W), GELU between layers."""
    h = x[..., None]
    for layer, (w, b) in enumerate(zip(*net)):
        h = _convolution(h, w, b)
        if layer < len(net[0]) - 1:
            h = torch.nn.functional.gelu(h)
    return h[..., 0]


def _exact_train(case, seed):
    x, y = _train_batch(case, seed)
    w, b = _network_arrays(seed)
    for t in w + b:
        t.requires_grad_()
    loss = ((_network((w, b), x[..., 0].double()) - y.double()) ** 2).mean()
    grads = torch.autograd.grad(loss, w + b)
    grads_w, grads_b = list(grads[: len(w)]), list(grads[len(w):])

    def padded(t, layer, weights):
        """The framework's padded layouts: (32, 25, 8 or 32) and (32,)."""
        shape = (32, 25, 8 if layer == 0 else 32) if weights else (32,)
        out = torch.zeros(shape, dtype=torch.float64, device="cuda")
        out[tuple(slice(0, m) for m in t.shape)] = t
        return out

    def updated(t, g):
        # first Adam step: both moments bias-corrected to g and g^2
        return t.detach() - 1e-3 * g / (g.abs() + 1e-8)

    def pad(ts, weights):
        return [padded(t, layer, weights) for layer, t in enumerate(ts)]

    return (pad(grads_w, True), pad(grads_b, False),
            pad([updated(t, g) for t, g in zip(w, grads_w)], True),
            pad([updated(t, g) for t, g in zip(b, grads_b)], False))


def _exact_les(case, seed):
    w, b = _network_arrays(seed)
    w[0] = w[0] / LES_IN
    w[-1], b[-1] = w[-1] * LES_OUT, b[-1] * LES_OUT
    return _exact_step(_les_step(case), seed, net=(w, b))


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _exact_step(case, seed)
    if kind == "ensemble":
        return _exact_ensemble(case, seed)
    if kind == "transform":
        x = _transform_input(case, seed).double()
        return torch.fft.rfftn(x, dim=(-3, -2, -1), norm="forward"), x
    if kind == "outputs":
        return _exact_outputs(case, seed)
    if kind == "train":
        return _exact_train(case, seed)
    return _exact_les(case, seed)

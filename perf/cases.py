"""The calls whose time this framework is judged by, from the 40 x 1 x 40 example
runs to the 512 x 512 x 128 mixed-precision production run.

A case's "kind" says which public entry points a pass goes through:

step          State.step over a few time steps of a run in progress, between
              the host copies of a restart: the predictands of a stored record
              are written to the state (pcf_set_field), the steps are taken,
              and the predictands are read back (pcf_get_field) into pinned
              buffers and stored in FP32, as output.record_datasets stores
              them.  A pass therefore always covers the same steps; where a
              solve starts from the previous steps' solutions there are enough
              of them that no step is its own predecessor.  The Exner pressure
              is defined up to a constant outside the compressible model; its
              mean is taken out of the record there.
ensemble      the same for several members that share the GPU, each stepped by
              its own thread with its solves in a SolveBatch, as ensemble()
              runs them.
net_forward   pcf_net_forward of the learned guess's network on device vectors.
net_gradients pcf_net_gradients: forward, loss and all parameter gradients.
"""
import ctypes
import dataclasses
import math
import threading

import numpy as np
import torch

import __graft_entry__

LAYERS = (3, 32, 32, 32, 32, 32, 1)  # channels of the network


def _step(name, setup, nx, ny, nz, steps, **options):
    case = {"name": name, "kind": "step", "setup": setup, "nx": nx, "ny": ny, "nz": nz, "steps": steps,
            "model": "PseudoIncompressible", "tracer": False, "precision": "fp64", "preconditioner": "line_relaxation",
            "storage": "fp32", "guess": "zero", "flux": "fp64"}
    case.update(options)
    return case


MULTIGRID = {"precision": "mixed", "preconditioner": "multigrid", "storage": "bf16", "guess": "previous", "flux": "mixed"}


def listed():
    return [
        # the examples' own size (the test-suite's runs, quick looks): launches and latency
        _step("hill_40x1x40", "periodic_hill", 40, 1, 40, 4, model="Boussinesq"),
        # a two-dimensional bubble study of the compressible model
        _step("bubble_96x1x128", "hot_bubble", 96, 1, 128, 4, model="Compressible"),
        # ragged sizes: an odd x, nothing a multiple of a tile
        _step("hills_75x53x41", "hills", 75, 53, 41, 3),
        # the compressible equations with a passive tracer, FP64
        _step("tracer_120x96x72", "hills", 120, 96, 72, 2, model="Compressible", tracer=True),
        # FP32 line relaxation at a medium size, reference flux arithmetic
        _step("line32_128x128x64", "hills", 128, 128, 64, 2, precision="mixed", guess="previous"),
        # a desktop-sized multigrid run
        _step("mg_96x80x64", "hills", 96, 80, 64, 4, **MULTIGRID),
        # the headline configuration: the reference's method in FP64
        _step("wave_256x256x128", "hills", 256, 256, 128, 1),
        # the headline configuration in mixed precision with the multigrid preconditioner
        _step("mg_256x256x128", "hills", 256, 256, 128, 3, **MULTIGRID),
        # the mixed-precision production run over many hills, the largest state
        _step("mg_512x512x128", "hills", 512, 512, 128, 2, **MULTIGRID),
        # seeded bubble members of uneven sizes sharing the GPU
        {"name": "ensemble_10", "kind": "ensemble", "members": 10, "steps": 2, "precision": "mixed"},
        # the learned guess at the headline size: one forward per solve
        {"name": "net_forward_256x256x128", "kind": "net_forward", "nx": 256, "ny": 256, "nz": 128},
        # a training step's gradients on a training-run size
        {"name": "net_gradients_128x128x64", "kind": "net_gradients", "nx": 128, "ny": 128, "nz": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["plane", "fp64", "fp64", "line32", "multigrid", "multigrid", "ensemble", "net_forward",
                       "net_gradients"])
    if kind == "plane":  # the two-dimensional examples
        setup = rng.choice(["periodic_hill", "hot_bubble", "cold_bubble"])
        model = {"periodic_hill": "Boussinesq", "hot_bubble": "Compressible"}.get(setup, "PseudoIncompressible")
        nx = _log_int(rng, 32, 320)
        case = _step("", setup, nx, 1, max(24, int(nx * rng.uniform(0.8, 1.4))), rng.randint(2, 5), model=model)
    elif kind == "fp64":  # the reference's method, any size and parity
        nx, ny, nz = _log_int(rng, 24, 224), _log_int(rng, 24, 224), _log_int(rng, 24, 128)
        compressible = rng.random() < 0.3
        case = _step("", "hills", nx, ny, nz, 1 if nx * ny * nz > 1500000 else 2,
                     model="Compressible" if compressible else "PseudoIncompressible",
                     tracer=compressible and rng.random() < 0.5)
    elif kind == "line32":
        nx, ny, nz = 2 * _log_int(rng, 12, 96), _log_int(rng, 24, 192), _log_int(rng, 24, 112)
        case = _step("", "hills", nx, ny, nz, 2, precision="mixed", storage=rng.choice(["fp32", "bf16"]),
                     guess=rng.choice(["zero", "previous"]), flux=rng.choice(["fp64", "mixed"]))
    elif kind == "multigrid":  # sizes that aggregate a few times, as such runs are set up
        nx, ny, nz = 16 * _log_int(rng, 2, 20), 16 * _log_int(rng, 2, 20), 4 * _log_int(rng, 8, 32)
        guess = rng.choice(["zero", "previous", "extrapolated"])
        case = _step("", "hills", nx, ny, nz, {"zero": 1, "previous": 2, "extrapolated": 3}[guess], precision="mixed",
                     preconditioner="multigrid", storage=rng.choice(["fp32", "bf16", "bf16"]), guess=guess,
                     flux=rng.choice(["fp64", "mixed"]))
    elif kind == "ensemble":
        return {"kind": "ensemble", "members": rng.randint(4, 12), "steps": rng.randint(1, 3),
                "precision": rng.choice(["fp64", "mixed"])}
    else:
        top = 8 if kind == "net_forward" else 6
        return {"kind": kind, "nx": 32 * rng.randint(1, top), "ny": _log_int(rng, 24, 32 * top),
                "nz": _log_int(rng, 16, 128 if kind == "net_forward" else 96)}
    del case["name"]
    return case


# ---- states ------------------------------------------------------------------

def _namelists(pcf, case, seed):
    rng = np.random.default_rng(seed)
    ex = pcf.examples
    nx, ny, nz, setup = case["nx"], case["ny"], case["nz"], case["setup"]
    if setup == "periodic_hill":
        nl = ex.periodic_hill(x_size=nx, z_size=nz)
        nl.atmosphere.initial_u = float(rng.uniform(9.0, 11.0))
    elif setup in ("hot_bubble", "cold_bubble"):
        sign = -1.0 if setup == "hot_bubble" else 1.0
        nl = getattr(ex, setup)(x_size=nx, z_size=nz)
        nl.atmosphere.initial_rhop = dataclasses.replace(nl.atmosphere.initial_rhop,
                                                         amplitude=sign * float(rng.uniform(0.004, 0.006)))
    else:
        nl = ex.gaussian_hills_3d(x_size=nx, y_size=ny, z_size=nz, seed=seed, n_hills=4 if nx < 512 else 16,
                                  precision=case["precision"])
        nl.atmosphere.model = case["model"]
    if case["tracer"]:
        d = nl.domain
        nl.tracer = pcf.TracerNamelist(tracer_setup="TracerOn", initial_tracer=pcf.TracerDipole(d.lx / 4, d.ly / 4))
    p = nl.poisson
    p.precision, p.preconditioner_type = case["precision"], case["preconditioner"]
    p.preconditioner_storage, p.initial_guess = case["storage"], case["guess"]
    p.mg_coarse_steps = 2
    nl.discretization.flux_precision = case["flux"]
    nl.output.output_steps, nl.output.iterations, nl.output.tmax = True, 1 << 20, 1.0e9
    return nl


class _Run:
    """A run in progress and the record it continues from, in pinned memory."""

    def __init__(self, pcf, nl, warm_steps):
        self.pcf, self.st = pcf, pcf.State(nl)
        if nl.poisson.initial_cleaning:
            self.st.initial_cleaning()
        for _ in range(warm_steps):
            self.st.step()
        self.names = ["RHO", "RHOP", "U", "V", "W", "PIP"]
        self.names += ["P"] if nl.atmosphere.model == "Compressible" else []
        self.names += ["CHI"] if nl.tracer.tracer_setup == "TracerOn" else []
        shape = (len(self.names), self.st.nzz, self.st.nyy, self.st.nxx)
        self.start = torch.empty(shape, dtype=torch.float64, pin_memory=True)
        self.end = torch.empty(shape, dtype=torch.float64, pin_memory=True)
        self.record = torch.empty(shape, dtype=torch.float32)
        self.time = self.st.time()[0]
        self._copy("pcf_get_field", self.start)

    def _copy(self, call, buffers):
        for name, b in zip(self.names, buffers):
            p = ctypes.cast(b.data_ptr(), ctypes.POINTER(ctypes.c_double))
            rc = getattr(self.st.lib, call)(self.st.h, self.pcf._abi.FIELD[name], p)
            if rc:
                raise self.pcf.PinCFlowError(rc, self.st.lib.pcf_last_error().decode())

    def advance(self, steps):
        st = self.st
        self._copy("pcf_set_field", self.start)
        if "P" in self.names:
            st.synchronize_compressible_atmosphere()
        st.lib.pcf_set_time(st.h, self.time)
        for _ in range(steps):
            st.step()
        self._copy("pcf_get_field", self.end)
        if "P" not in self.names:  # the Neumann problem leaves the Exner pressure's constant to the iteration
            self.end[5] -= self.end[5].mean()
        self.record.copy_(self.end)
        return {name: r for name, r in zip(self.names, self.record)}


# ---- the network ---------------------------------------------------------------

def _net_inputs(case, seed):
    """Parameters, and smooth fields with noise as the right-hand side, the
    warm start and the terrain channel of the network's input look."""
    rng = np.random.default_rng(seed)
    parts = []
    for cin, cout in zip(LAYERS[:-1], LAYERS[1:]):
        parts += [rng.standard_normal(27 * cout * cin) * math.sqrt(2.0 / (27 * cin)), 0.05 * rng.standard_normal(cout)]
    params = np.concatenate(parts).astype(np.float32)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    at = torch.arange(nx, device="cuda") * (2.0 * math.pi / nx)
    wave = (torch.sin(at) + 0.5 * torch.cos(3.0 * at)).repeat(ny * nz)
    x = 0.7 * torch.randn((n, 3), device="cuda", generator=gen) + wave[:, None]
    x[:, 2] = 0.05 * wave.abs()
    target = 0.1 * torch.randn(n, device="cuda", generator=gen) + 0.1 * wave
    return params, x.float().contiguous(), target.float().contiguous()


def _net_exact(case, params, x):
    """The network in 64 bits on (nz, ny, nx, channels) arrays; params: the
    layers' (W[27][cout][cin], b[cout]) as torch tensors."""
    y = x.double().reshape(case["nz"], case["ny"], case["nx"], 3)
    for layer, (w, b) in enumerate(params):
        taps = None
        up = torch.nn.functional.pad(y, (0, 0, 0, 0, 0, 0, 1, 1))
        for t in range(27):
            dx, dy, dz = t % 3 - 1, t // 3 % 3 - 1, t // 9 - 1
            shifted = torch.roll(up[1 + dz:1 + dz + case["nz"]], (-dy, -dx), (1, 2))
            part = shifted.reshape(-1, w.shape[2]) @ w[t].T.contiguous()
            taps = part if taps is None else taps + part
        y = (taps + b).reshape(*y.shape[:3], w.shape[1])
        if layer < 5:
            y = 0.5 * y * (1.0 + torch.erf(y / math.sqrt(2.0)))
    return y.reshape(-1)


def _split(params):
    out, at = [], 0
    for cin, cout in zip(LAYERS[:-1], LAYERS[1:]):
        nw = 27 * cout * cin
        w = torch.tensor(params[at:at + nw], dtype=torch.float64, device="cuda").reshape(27, cout, cin)
        out.append((w, torch.tensor(params[at + nw:at + nw + cout], dtype=torch.float64, device="cuda")))
        at += nw + cout
    return out


# ---- the interface -------------------------------------------------------------

def prepare(case, seed):
    pcf = __graft_entry__.load_package()
    if case["kind"] == "step":
        return {"case": case, "run": _Run(pcf, _namelists(pcf, case, seed), 2)}
    if case["kind"] == "ensemble":
        sizes = [(64, 64), (96, 64), (64, 96), (128, 64), (96, 96)]
        runs = []
        for m in range(case["members"]):
            nx, nz = sizes[m % len(sizes)]
            nl = pcf.examples.bubble_member(seed=1000 * (seed % 1000) + m, x_size=nx, z_size=nz,
                                            precision=case["precision"])
            if case["precision"] == "mixed":
                nl.discretization.flux_precision = "mixed"
            runs.append(_Run(pcf, nl, 1))
        return {"case": case, "pcf": pcf, "runs": runs}
    params, x, target = _net_inputs(case, seed)
    training = case["kind"] == "net_gradients"
    net = pcf.learned.GuessNetwork(case["nx"], case["ny"], case["nz"], training=training, params=params)
    state = {"case": case, "pcf": pcf, "net": net, "x": x, "target": target,
             "y": torch.empty(x.shape[0], dtype=torch.float32, device="cuda"),
             "grads": torch.empty(net.n_params, dtype=torch.float32, pin_memory=True)}
    torch.cuda.synchronize()
    return state


def _run_ensemble(state):
    batch = state["pcf"].SolveBatch()
    runs, steps = state["runs"], state["case"]["steps"]
    out, errors = [None] * len(runs), []

    def member(m):
        try:
            batch.attach(runs[m].st)
            try:
                out[m] = runs[m].advance(steps)
            finally:
                batch.detach(runs[m].st)
        except Exception as e:
            errors.append(e)

    threads = [threading.Thread(target=member, args=(m,)) for m in range(len(runs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    batch.close()
    if errors:
        raise errors[0]
    return [r.record for r in runs]


def run(state):
    kind = state["case"]["kind"]
    if kind == "step":
        return state["run"].advance(state["case"]["steps"])
    if kind == "ensemble":
        return _run_ensemble(state)
    net = state["net"]
    x = ctypes.c_void_p(state["x"].data_ptr())
    if kind == "net_forward":
        rc = net.lib.pcf_net_forward(net.h, x, ctypes.c_void_p(state["y"].data_ptr()))
        out = state["y"]
    else:
        loss = ctypes.c_double(0.0)
        grads = ctypes.cast(state["grads"].data_ptr(), ctypes.POINTER(ctypes.c_float))
        rc = net.lib.pcf_net_gradients(net.h, x, ctypes.c_void_p(state["target"].data_ptr()), grads,
                                       ctypes.byref(loss))
        out = {"grads": state["grads"], "loss": torch.tensor(loss.value, dtype=torch.float32)}
    if rc:
        raise state["pcf"].PinCFlowError(rc, net.lib.pcf_last_error().decode())
    return out


def exact(case, seed):
    """The network's results in 64 bits (its parameters, input and target are
    FP32); a time step has no closed form."""
    if case["kind"] not in ("net_forward", "net_gradients"):
        return None
    params, x, target = _net_inputs(case, seed)
    layers = _split(params)
    if case["kind"] == "net_forward":
        with torch.no_grad():
            return _net_exact(case, layers, x)
    flat = [p.requires_grad_(True) for layer in layers for p in layer]
    loss = ((_net_exact(case, layers, x) - target.double()) ** 2).mean()
    grads = torch.autograd.grad(loss, flat)
    return {"grads": torch.cat([g.reshape(-1) for g in grads]), "loss": None}


def work(case):
    """A step: every predictand read and written once, and the static
    background, metric and sponge fields (ten) read once, FP64; one operator
    application's arithmetic per cell for each of its two solves and of the
    order of 500 operations of fluxes and updates.  The network: its FP32
    input, output and parameters, and its multiply-adds (three times as many
    with the gradients)."""
    if case["kind"] == "step":
        n = case["nx"] * case["ny"] * case["nz"]
        fields = 6 + (case["model"] == "Compressible") + case["tracer"]
        return {"bytes": 8.0 * n * (2 * fields + 10) * case["steps"], "flops": 600.0 * n * case["steps"]}
    if case["kind"] == "ensemble":
        sizes = [(64, 64), (96, 64), (64, 96), (128, 64), (96, 96)]
        n = sum(sizes[m % 5][0] ** 2 * sizes[m % 5][1] for m in range(case["members"]))
        return {"bytes": 8.0 * n * 22 * case["steps"], "flops": 600.0 * n * case["steps"]}
    n = case["nx"] * case["ny"] * case["nz"]
    macs = n * 27 * sum(a * b for a, b in zip(LAYERS[:-1], LAYERS[1:]))
    count = sum(27 * a * b + b for a, b in zip(LAYERS[:-1], LAYERS[1:]))
    return {"bytes": 16.0 * n + 4.0 * count, "flops": 2.0 * macs * (3 if case["kind"] == "net_gradients" else 1)}

"""What this framework's users have it do, as cases to time.

A case is a dict of plain values whose "what" names the work:

  lag       a pure-cell Lagrangian run on the device (BookLeaf.run, run_graph):
            Sod, Sedov, Taylor-Green, Noh, a JWL column driving a Tait liquid;
            with the anti-hourglass, sub-zonal pressure and mid-length options
  eul       the same with the Eulerian remap every step
  mixed     two-material Sod with mixed interface cells, Eulerian
  relax     two-material Sod with ALE node relaxation as the mesh motion
  learned   the same mesh motion proposed by the node-relaxation network
  ensemble  many Sod/Sedov instances stepped together (Ensemble.run)
  records   a Lagrangian run with the per-step tables (set_diagnostics), read
            back at its end
  drivers   the reference's solver sequence driver by driver (getdt, lagstep,
            alestep), as a host that keeps its own step loop calls them
  train     Adam steps of the node-relaxation network on stored pairs

A pass of the mesh workloads rewinds the device fields to a state the program
kept (device copies of the fields a step reads, through their device
pointers), runs a fixed number of steps and returns the fields on the device
with the dt history: a program that runs many batches from one start.  The
state it rewinds to is `warm` steps into the run, so that the flow is under
way.  Inputs come from the seed: the seed scales the initial density and
energy, and gives the ensemble's states, the network and the training pairs;
sizes come from the case alone.
"""
import math

import numpy as np
import torch

from bookleaf_f90_amd import abi
from bookleaf_f90_amd import problem as P
from bookleaf_f90_amd.device import BookLeaf, Ensemble, RelaxNet

# fields a step reads (and a pass rewinds), by what steps them
NODES = ("ndx", "ndy", "ndu", "ndv")
ELEMENTS = ("eldensity", "elenergy", "elpressure", "elcs2")
REMAP = ("elmass", "cnmass")
GEOMETRY = ("cnx", "cny", "a1", "a2", "a3", "b1", "b2", "b3", "cnwt", "elvolume")
COMPONENTS = ("cpdensity", "cpenergy", "cppressure", "cpcs2", "cpvolume", "cpa1", "cpa3",
              "cpb1", "cpb3")


def listed():
    return [
        # the smallest run in use: the 200x20 Sod tube to t = 0.2 (395 steps
        # at the default controls), where launches and latency count
        dict(name="sod_200x20", what="lag", flow="sod", nx=200, ny=20, steps=395, warm=0),
        # the reference's own small Eulerian deck size
        dict(name="sod_eul_100x25", what="eul", flow="sod", nx=100, ny=25, steps=120, warm=20),
        # the headline blast: most of the mesh at rest, hourglass control on
        dict(name="sedov_1024", what="lag", flow="sedov", nx=1024, ny=1024, jitter=0.1,
             steps=60, warm=150),
        # every element in motion, a size that is no power of two
        dict(name="tgv_700", what="lag", flow="tgv", nx=700, ny=700, steps=40, warm=10),
        # the headline remap: two materials, mixed interface cells, Eulerian
        dict(name="mixed_2048x256", what="mixed", nx=2048, ny=256, steps=40, warm=100),
        # pure cells with the remap on an odd mesh, everything in motion
        dict(name="sedov_eul_401", what="eul", flow="sedov", nx=401, ny=401, steps=60, warm=60),
        # ALE with node relaxation (2 EQUI sweeps)
        dict(name="relax_1024x512", what="relax", nx=1024, ny=512, steps=30, warm=30, sweeps=2,
             om=0.5),
        # the network's mesh motion in place of 8 EQUI sweeps
        dict(name="learned_512x256", what="learned", nx=512, ny=256, steps=60, warm=20,
             sweeps=8, om=0.25),
        # an ensemble of uneven meshes
        dict(name="ensemble_48", what="ensemble", instances=48, nmin=64, nmax=256, sizes=2025,
             steps=20, warm=40),
        # a run recorded every step
        dict(name="records_sedov_512", what="records", flow="sedov", nx=512, ny=512, steps=150,
             warm=60),
        # the drop-in boundary: one call per reference driver
        dict(name="drivers_sedov_512", what="drivers", flow="sedov", nx=512, ny=512, steps=5,
             warm=20, eulerian=False),
        # training the network: the recipe's batch
        dict(name="train_8192", what="train", pairs=200000, batch=8192, steps=20),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["lag", "lag", "lag", "eul", "eul", "mixed", "relax", "learned",
                       "ensemble", "records", "drivers", "drivers", "train"])
    if what == "train":
        return dict(what=what, pairs=_log(rng, 20000, 400000), batch=_log(rng, 500, 20000),
                    steps=rng.randint(5, 20))
    if what == "ensemble":
        nmin = rng.randint(24, 100)
        return dict(what=what, instances=_log(rng, 2, 80), nmin=nmin,
                    nmax=rng.randint(nmin + 8, 200), sizes=rng.randint(1, 1 << 20),
                    steps=rng.randint(5, 20), warm=rng.randint(0, 40))
    nel = _log(rng, 800, 300000)
    aspect = math.exp(rng.uniform(0.0, math.log(8.0)))
    if what in ("relax", "learned"):
        nel = max(nel, 4000)
        aspect = min(aspect, 3.0)
    nx = max(8, int(round(math.sqrt(nel * aspect))))
    ny = max(6, int(round(nx / aspect)))
    steps = max(5, min(200, int(1.0e7 / (nx * ny))))
    case = dict(what=what, nx=nx, ny=ny, steps=steps, warm=rng.randint(0, 60))
    if what in ("lag", "eul", "records", "drivers"):
        case["flow"] = rng.choice(["sod", "sod", "sedov", "tgv", "noh"]
                                  + (["tait_jwl"] if what == "lag" else []))
        if case["flow"] in ("sedov", "tgv", "noh"):
            case["nx"] = case["ny"] = max(12, int(round(math.sqrt(nel))))
            case["steps"] = max(5, min(200, int(1.0e7 / case["nx"] ** 2)))
        case["option"] = rng.choice(["plain", "plain", "hourglass", "subzonal", "midlength"]
                                    if case["flow"] == "sod" else ["plain"])
    if what in ("eul", "drivers"):
        case["warm"] = min(case["warm"], 30)
    if what == "drivers":
        case["eulerian"] = rng.random() < 0.5
        case["steps"] = max(2, case["steps"] // 8)
    if what in ("relax", "learned"):
        case["sweeps"] = rng.choice([1, 2, 3, 4, 8])
        case["om"] = rng.choice([0.25, 0.5]) if case["sweeps"] <= 3 else 0.25
        case["steps"] = min(case["steps"], 60)
        case["warm"] = min(case["warm"], 20)
    return case


def work(case):
    """The state a step reads once and writes once, over the pass's steps.
    Lagrangian: connectivity, material and region 24, rho, e, p, cs2 read and
    written 64, mass and corner masses 40, at-rest flags 2 per element;
    positions and velocities read and written 64, type 4 per node.  A remap
    writes mass and corner masses too (40).  The operation counts are those
    of the step's formulas (about 900 FP64 operations an element for an
    element in motion, 700 more for the remap)."""
    n = case["steps"]
    if case["what"] == "train":
        # forward, input gradients, weight gradients: 26x64 + 64x64 + 64x2
        return {"bytes": n * (4.0 * 28 * case["batch"] + 7 * 4.0 * abi.MLP_NPARAM),
                "flops": n * 3 * 2.0 * 5888 * case["batch"]}
    if case["what"] == "ensemble":
        nel = sum(q["nx"] * q["ny"] for q in _members(case))
        nnd = sum((q["nx"] + 1) * (q["ny"] + 1) for q in _members(case))
    else:
        nel, nnd = case["nx"] * case["ny"], (case["nx"] + 1) * (case["ny"] + 1)
    if case["what"] == "drivers":
        # the drivers' own inputs and outputs
        e, d, f = (2168, 380, 1600) if case["eulerian"] else (1664, 272, 900)
        return {"bytes": float(n * (e * nel + d * nnd)), "flops": float(n * f * nel)}
    remap = case["what"] in ("eul", "mixed", "relax", "learned")
    return {"bytes": float(n * ((170 if remap else 130) * nel + 68 * nnd)),
            "flops": float(n * (1600 if remap else 900) * nel)}


# ---- what a program has in hand -------------------------------------------

def _members(case):
    return P.ensemble_params(case["instances"], seed=case["sizes"], nmin=case["nmin"],
                             nmax=case["nmax"])


def _scale(p, rng):
    """Another state of the same flow: density and energy scaled."""
    a, b = rng.uniform(0.9, 1.1, size=2)
    p.density = p.density * a
    p.energy = p.energy * b
    if p.ncp:
        p.cpdensity = p.cpdensity * a
        p.cpenergy = p.cpenergy * b
    return p


def _problem(case, rng):
    what, nx, ny = case["what"], case["nx"], case["ny"]
    if what == "mixed":
        return _scale(P.sod2mat_mixed(nx=nx, ny=ny), rng)
    if what in ("relax", "learned"):
        p = P.sod2mat_mixed(nx=nx, ny=ny, eulerian=False, jitter=0.1, seed=2024)
        return _scale(P.with_relaxation(p, abi.RELAX_EQUI, nsweep=case["sweeps"],
                                        om=case["om"]), rng)
    flow = case["flow"]
    if flow == "sod":
        p = P.sod(nx=nx, ny=ny, height=ny / nx, time_end=1.0e30)
        option = case.get("option", "plain")
        if option == "hourglass":
            p.kappareg[:] = 0.01
        elif option == "subzonal":
            p.pmeritreg[:] = 0.1
        elif option == "midlength":
            p.zmidlength[:] = 1
    elif flow == "sedov":
        p = P.sedov(n=nx, jitter=case.get("jitter", 0.0), kappa=0.01)
    elif flow == "tgv":
        p = P.taylor_green(n=nx)
    elif flow == "noh":
        p = P.noh(n=nx, time_end=1.0e30)
    else:
        p = P.tait_jwl(nx=nx, ny=ny)
    if what == "eul" or case.get("eulerian"):
        p.config["zeul"] = 1
    p.__post_init__()
    if flow == "tait_jwl":  # the liquid stays at its reference density
        p.energy = p.energy * rng.uniform(0.9, 1.1)
        return p
    return _scale(p, rng)


class _Device:
    """A field's device memory as torch takes it.  It holds the handle, and a
    tensor made of it holds it: the memory stays until the last tensor over
    it is gone."""

    def __init__(self, handle, ptr, count):
        self.handle = handle
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": "<f8", "version": 3,
                                         "data": (ptr, False)}


class _Fields:
    """The handle's device fields as tensors (the fields of a run swap
    buffers, so the pointer is asked for each time)."""

    def __init__(self, handle):
        self.handle, self.known = handle, {}
        self.count = {}

    def __call__(self, name):
        ptr = self.handle.device_ptr(name)
        t = self.known.get((ptr, name))
        if t is None:
            if name not in self.count:
                self.count[name] = self.handle._info(name)[1]
            t = torch.as_tensor(_Device(self.handle, ptr, self.count[name]), device="cuda")
            t.handle = self.handle
            self.known[(ptr, name)] = t
        return t


def _weights(rng):
    """He-uniform weights of the 26-64-64-2 network, small biases."""
    parts = []
    for rows, cols in ((64, 26), (64, 64), (2, 64)):
        a = math.sqrt(6.0 / cols)
        parts += [rng.uniform(-a, a, rows * cols), rng.uniform(-0.01, 0.01, rows)]
    return np.concatenate(parts).astype(np.float32)


def _network(rng):
    """A network whose output is a small correction to one plain sweep (in
    units of the cell width), as a trained one's is."""
    net = RelaxNet(seed=0)
    net.set_weights(_weights(rng))
    one = np.ones(abi.MLP_NIN, np.float32)
    net.set_norm(0.0 * one, one, np.zeros(2, np.float32), np.full(2, 1.0e-4, np.float32))
    return net


def _pairs(n, rng):
    """Training pairs: stencil features, and displacements near one sweep's
    (the last two features)."""
    x = rng.standard_normal((n, abi.MLP_NIN)).astype(np.float32)
    x[:, 24:] *= 0.01
    t = (x[:, 24:] + 0.002 * np.tanh(x[:, :2] * x[:, 2:4])).astype(np.float32)
    return x, t


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    what = case["what"]
    state = {"case": case}
    if what == "train":
        x, t = _pairs(case["pairs"], rng)
        net = RelaxNet(seed=0, capacity=len(x))
        net.add_pairs(x, t)
        net.normalize()
        state.update(net=net, start=_weights(rng))
        return state
    if what == "ensemble":
        params = _members(case)
        for q in params:
            f = float(rng.uniform(0.9, 1.1))
            q["e_l"] *= f
            q["e_r"] *= f
        handle = Ensemble(params)
        if case["warm"]:
            handle.run(case["warm"])
        names, out = NODES + ELEMENTS, NODES + ELEMENTS
    else:
        handle = BookLeaf(_problem(case, rng))
        names, out = NODES + ELEMENTS, NODES + ELEMENTS + ("elvolume",)
        if what in ("eul", "mixed", "relax", "learned") or case.get("eulerian"):
            names, out = names + REMAP, out + REMAP
        if handle.problem.ncp:
            names, out = names + COMPONENTS, out + COMPONENTS[:5]
        if what == "drivers":
            names = names + GEOMETRY
        if what == "learned":
            state["net"] = _network(rng)
            handle.relax_learned(state["net"])
        if case["warm"]:
            handle.run(case["warm"], runner="run_graph")
    fields = _Fields(handle)
    handle.synchronize()
    state.update(handle=handle, fields=fields, out=out,
                 kept={n: fields(n).clone() for n in names})
    if what != "ensemble":
        ts = handle.ts
        state["ts"] = (ts.time, ts.dt, ts.dts, ts.nstep, ts.idtel, ts.sdt)
    torch.cuda.synchronize()
    return state


def run(state):
    case = state["case"]
    what, n = case["what"], case["steps"]
    if what == "train":
        net = state["net"]
        net.set_weights(state["start"])
        loss = net.train(n, batch=case["batch"], lr=1.0e-3, seed=5)
        return {"loss": loss, "weights": net.weights()}
    handle, fields, kept = state["handle"], state["fields"], state["kept"]
    torch._foreach_copy_([fields(k) for k in kept], list(kept.values()))
    torch.cuda.current_stream().synchronize()  # the handle steps on a stream of its own
    if what != "ensemble":
        ts = handle.ts
        ts.time, ts.dt, ts.dts, ts.nstep, ts.idtel, ts.sdt = state["ts"]
    if what == "ensemble":
        history = handle.run(n)
    elif what == "drivers":
        history = []
        for _ in range(n):
            handle.step()
            history.append((ts.dt, float(ts.idtel), float(ts.sdt)))
        history = np.array(history)
    elif what == "records":
        handle.set_diagnostics(True, maxrec=n)
        history = handle.run(n, runner="run_graph")
        history = list(history) + list(handle.diagnostics().values())
    else:
        history = handle.run(n, runner="run_graph")
    if what == "drivers":
        handle.synchronize()  # the last drivers' kernels are on the handle's stream
    return {"history": history, "fields": {k: fields(k) for k in state["out"]}}


# ---- in 64 bits -------------------------------------------------------------
# The hydrodynamics computes and returns 64-bit numbers throughout, in the
# reference's order of operations: its start's own outputs are what there is
# to compare with.  The network's training is 32-bit sums over BF16-rounded
# operands; this is the same training with 64-bit sums.

def _bf16(a):
    return torch.from_numpy(np.asarray(a, np.float32)).bfloat16().double()


def _drawn(seed, it, batch, npairs):
    """The pairs of Adam step `it`: a counter hash of (seed, step, place)."""
    mask = (1 << 64) - 1

    def mix(z):
        z = (z + np.uint64(0x9e3779b97f4a7c15))
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xbf58476d1ce4e5b9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94d049bb133111eb)
        return z ^ (z >> np.uint64(31))

    with np.errstate(over="ignore"):
        place = np.uint64((it << 32) & mask) | np.arange(batch, dtype=np.uint64)
        return (mix(np.uint64(seed) ^ mix(place)) % np.uint64(npairs)).astype(np.int64)


def exact(case, seed):
    if case["what"] != "train":
        return None
    rng = np.random.default_rng(seed)
    x, t = _pairs(case["pairs"], rng)
    w = _weights(rng)
    x64 = x.astype(np.float64)
    mu, sd = x64.mean(0), x64.std(0)
    r = (t - x[:, 24:]).astype(np.float64)
    mu_t, sd_t = r.mean(0).astype(np.float32), r.std(0).astype(np.float32)
    xn = _bf16((x - mu.astype(np.float32)) * (1.0 / sd).astype(np.float32))
    target = torch.from_numpy(((t - x[:, 24:]) - mu_t) / sd_t).double()
    shapes = ((64, 26), (64,), (64, 64), (64,), (2, 64), (2,))
    sizes = [int(np.prod(s)) for s in shapes]
    w = torch.from_numpy(w.astype(np.float64))
    m, v = torch.zeros_like(w), torch.zeros_like(w)
    b1, b2 = float(np.float32(0.9)), float(np.float32(0.999))
    batch, loss = case["batch"], []
    for it in range(case["steps"]):
        at = torch.from_numpy(_drawn(5, it, batch, len(x)))
        a0, y0 = xn[at], target[at]
        W1, c1, W2, c2, W3, c3 = (p.reshape(s) for p, s in zip(w.split(sizes), shapes))
        W1, W2, W3 = (_bf16(q.numpy()) for q in (W1, W2, W3))
        z1 = a0 @ W1.T + c1
        a1 = _bf16(z1.clamp(min=0.0).numpy())
        z2 = a1 @ W2.T + c2
        a2 = _bf16(z2.clamp(min=0.0).numpy())
        e = a2 @ W3.T + c3 - y0
        loss.append(float((e * e).sum() / (2 * batch)))
        d3 = e / batch
        d2 = (d3 @ W3) * (z2 > 0)
        d1 = (d2 @ W2) * (z1 > 0)
        g = torch.cat([(d1.T @ a0).reshape(-1), d1.sum(0), (d2.T @ a1).reshape(-1), d2.sum(0),
                       (d3.T @ a2).reshape(-1), d3.sum(0)])
        m = b1 * m + (1.0 - b1) * g
        v = b2 * v + (1.0 - b2) * g * g
        mh, vh = m / (1.0 - b1 ** (it + 1)), v / (1.0 - b2 ** (it + 1))
        w = w - float(np.float32(1.0e-3)) * mh / (vh.sqrt() + 1.0e-8)
    return {"loss": np.array(loss), "weights": w.numpy()}

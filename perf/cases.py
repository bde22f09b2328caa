"""Performance cases of the SPH step, the batched scenes and the learned closure.

Every case calls the package's public entry points as a simulation program does: a context is set
up once (scene uploaded, variants tuned where the program tunes), and a pass is the call that such a
program repeats.  Inputs are made here from the seed alone, so that `exact` can restate a pass in 64
bits without the package.

    listed()            the cases, smallest to largest
    draw(rng)           one more case of the same ranges
    prepare(case, seed) the state a program holds before the call
    run(state)          one pass and its outputs
    work(case)          the bytes and operations a pass cannot do without
    exact(case, seed)   what the pass returns, in 64 bits
"""
import ctypes as C
import math
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent.parent
WEIGHTS = ROOT / "watercube_amd" / "weights" / "closure.npy"

# The package's network: 195 inputs padded to 208, three hidden layers of 128, 3 outputs padded to 32.
NIN, NPAD, NH, NOUT, NOPAD = 195, 208, 128, 3, 32
SHAPES = [(NPAD, NH), (NH,), (NH, NH), (NH,), (NH, NH), (NH,), (NH, NOPAD), (NOPAD,)]
G = 9.81


# ---------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------
def _fluid(name, nx, ny, nz, fill, **kw):
    c = {"kind": "fluid", "nx": nx, "ny": ny, "nz": nz, "fill": fill, "ratio": 2.0, "constants": "dam_break",
         "ball": 0, "steps": 1, "tune": False, "wall": False, "mouse": False}
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the small scene of the fixtures (2,048 particles), one Fluid::update per frame: launches and latency
        _fluid("fluid_2k", 16, 16, 8, 0.48),
        # the 16,384-particle dam break run on for some steps per call, as a simulation without a viewer does
        _fluid("fluid_16k_8steps", 32, 32, 16, 0.48, steps=8),
        # the reference application's own default: 80,000 particles in a wide grid (about 20 a cell), cubic
        # equation of state, wall terms, the mouse ray held down, one update per frame
        _fluid("fluid_80k_reference", 44, 43, 43, 0.0175 * 44, ratio=0.04 / 0.0175, constants="reference",
               wall=True, mouse=True),
        # an odd block with sides that fit no tile, more neighbours than the usual spacing gives
        _fluid("fluid_193k_odd", 61, 47, 67, 0.67, ratio=2.3),
        # the million-particle block of the benchmark, tuned as the benchmark tunes it
        _fluid("fluid_1m", 100, 100, 100, 0.8, tune=True),
        # the largest scene: a 256^3 block and a falling ball of a million particles
        _fluid("fluid_17m", 256, 256, 256, 0.512, ball=1_000_000, tune=True),
        # independent scenes of 4,096 to 262,144 particles advanced together (a quarter of the benchmark's batch)
        {"name": "batch_64", "kind": "batch", "scenes": 64, "n_min": 4096, "n_max": 262144, "tune": True},
        # the step for callers that cannot allocate, on their own buffers
        {"name": "noalloc_216k", "kind": "noalloc", "nx": 60, "ny": 60, "nz": 60, "fill": 0.48, "ratio": 2.0},
        # the learned large step, judged, each particle's own correction: the benchmark's fastest method
        {"name": "closure_run_1m", "kind": "closure_run", "nx": 100, "ny": 100, "nz": 100, "fill": 0.8, "ratio": 2.0,
         "K": 8, "macro": 4, "smooth": False},
        # the closure network on inputs formed from the neighbour lists
        {"name": "closure_infer_262k", "kind": "closure_infer", "nx": 64, "ny": 64, "nz": 64, "fill": 0.512,
         "ratio": 2.0, "K": 4},
        # an epoch's slice of training: eight batches of 8,192 rows, then the parameters are read
        {"name": "train_8k", "kind": "train", "rows": 8192, "batches": 8},
        # loss and gradient over a validation split of a ragged size
        {"name": "gradient_51k", "kind": "gradient", "rows": 51_207},
    ]


def draw(rng):
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def sides(lo, hi):
        n = logint(lo, hi)
        a = max(4, round((n * rng.uniform(0.5, 2.0)) ** (1 / 3)))
        b = max(4, round((n / a * rng.uniform(0.7, 1.5)) ** 0.5))
        return {"nx": a, "ny": b, "nz": max(3, round(n / (a * b)))}

    kind = rng.choice(("fluid", "fluid", "fluid", "batch", "noalloc", "closure_run", "closure_infer", "train",
                       "gradient"))
    fill = round(rng.uniform(0.45, 0.8), 3)
    if kind == "fluid":
        return _fluid(None, fill=fill, ratio=round(rng.uniform(1.9, 2.35), 2), steps=rng.choice((1, 1, 3, 8)),
                      constants=rng.choice(("dam_break", "dam_break", "reference")), tune=rng.random() < 0.5,
                      wall=rng.random() < 0.3, mouse=rng.random() < 0.2, **sides(1500, 1_500_000))
    if kind == "batch":
        return {"kind": "batch", "scenes": logint(3, 64), "n_min": 1024 * rng.randint(1, 4),
                "n_max": logint(8192, 200_000), "tune": rng.random() < 0.5}
    if kind == "noalloc":
        return {"kind": "noalloc", "fill": round(rng.uniform(0.45, 0.55), 3), "ratio": 2.0, **sides(1500, 150_000)}
    if kind == "closure_run":
        return {"kind": "closure_run", "fill": fill, "ratio": 2.0, "K": rng.choice((2, 4, 8)),
                "macro": rng.randint(1, 4), "smooth": rng.random() < 0.5, **sides(16_000, 800_000)}
    if kind == "closure_infer":
        return {"kind": "closure_infer", "fill": fill, "ratio": rng.choice((2.0, 2.0, 2.2)), "K": rng.choice((2, 4, 8)),
                **sides(8000, 400_000)}
    if kind == "train":
        return {"kind": "train", "rows": logint(500, 9000), "batches": rng.randint(2, 8)}
    return {"kind": "gradient", "rows": logint(1000, 65_000)}


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _gen(seed):
    g = torch.Generator(device=_device())
    g.manual_seed(int(seed))
    return g


def _lattice(nx, ny, nz, s, jitter, gen, origin=(0.0, 0.0, 0.0), keep=None):
    """Records (n, 8) of a jittered lattice block, x fastest, with a smooth velocity field and a little noise;
    `keep` (count, centre): the lattice points nearest to a centre."""
    d = _device()
    i = torch.arange(nx * ny * nz, device=d)
    p = torch.stack([i % nx, (i // nx) % ny, i // (nx * ny)], 1).to(torch.float64).add_(0.5).mul_(s)
    p += torch.tensor(origin, device=d, dtype=torch.float64)
    if keep is not None:
        count, centre = keep
        r = (p - torch.tensor(centre, device=d, dtype=torch.float64)).square().sum(1)
        p = p[torch.argsort(r, stable=True)[:count].sort().values]
    n = len(p)
    rec = torch.zeros(n, 8, device=d)
    rec[:, :3] = p + (torch.rand(n, 3, generator=gen, device=d) * 2 - 1) * jitter
    rec[:, 4:7] = torch.randn(n, 3, generator=gen, device=d) * 0.05
    rec[:, 4] += 0.3 * torch.sin(9.0 * rec[:, 1])
    rec[:, 5] -= 0.2 * rec[:, 2]
    return rec


def _constants(case):
    """The scene's parameters as plain numbers (float32 values), primary fields first."""
    f = np.float32
    s = case["fill"] / max(case["nx"], case["ny"], case["nz"])
    h = f(case["ratio"] * s)
    reference = case.get("constants") == "reference"
    # the reference's own scene bins more widely than its kernel radius (h = 4 r, 21 bins in a unit cube for r = 0.01)
    R = max(1, int(math.floor(1.0 / float(h) * (0.84 if reference else 1.0) + 1e-4)))
    k = {"size": f(1.0), "R": R, "h": h, "bin": f(1.0) / f(R), "rho0": f(1000.0), "p0": f(0.0), "k": f(250.0),
         "mu": f(0.2), "m": f(1000.0 * s ** 3), "g": [0.0, -9.81, 0.0], "damping": f(0.5), "border": f(0.001),
         "vmax": f(50.0), "cubic": reference, "wall": bool(case.get("wall")), "mouse": bool(case.get("mouse")),
         "cam": [0.4, 0.4, 2.0], "dir": [0.02, -0.05, -0.9985], "dt": float(f(2e-4 * s / 0.015)), "s": s}
    if reference:
        k.update(rho0=f(500.0), k=f(100.0), mu=f(0.02), g=[0.0, -90.0, 0.0], damping=f(0.3), m=f(500.0 * s ** 3))
    return k


def _records(case, seed):
    gen, s = _gen(seed), _constants(case)["s"]
    rec = _lattice(case["nx"], case["ny"], case["nz"], s, 0.1 * s, gen)
    if case.get("ball"):
        side = int(2.2 * (case["ball"] * 3 / (4 * math.pi)) ** (1 / 3)) + 4
        low = [0.5 - side * s / 2, 0.8 - side * s / 2, 0.5 - side * s / 2]
        ball = _lattice(side, side, side, s, 0.1 * s, gen, low, (case["ball"], (0.5, 0.8, 0.5)))
        ball[:, 5] -= 2.0
        rec = torch.cat([rec, ball])
    return rec


def _batch_scenes(case, seed):
    """Plain cases of the batch's scenes, sizes from the case alone: blocks of varied sides."""
    rng = np.random.default_rng(case["scenes"] * 1_000_003 + case["n_max"])
    out = []
    for i in range(case["scenes"]):
        n = math.exp(rng.uniform(math.log(case["n_min"]), math.log(case["n_max"])))
        z = max(2, round((n / 4) ** (1 / 3)))
        x, y = ((2 * z, 2 * z), (z, 4 * z), (2 * z + 1, 2 * z - 1))[i % 3]
        out.append(({"nx": x, "ny": y, "nz": z, "fill": (0.48, 0.8, 0.5)[i % 3], "ratio": 2.0}, seed * 1000 + i))
    return out


def _numpy_records(rec):
    from watercube_amd import PARTICLE_DTYPE

    return rec.cpu().numpy().view(PARTICLE_DTYPE).reshape(-1)


def _params(case, n):
    """The package's parameter block of a case's constants."""
    from watercube_amd import _lib as L

    k = _constants(case)
    p = L.preset(L.WC_PRESET_REFERENCE_DEFAULT if k["cubic"] else L.WC_PRESET_DAM_BREAK_16K)
    p.num_particles, p.grid_res, p.size = n, k["R"], k["size"]
    p.kernel_radius, p.particle_mass, p.particle_radius = k["h"], k["m"], k["h"] / 4
    p.rest_density, p.rest_pressure, p.stiffness, p.viscosity = k["rho0"], k["p0"], k["k"], k["mu"]
    p.wall_damping, p.border, p.max_speed = k["damping"], k["border"], k["vmax"]
    p.eos = L.WC_EOS_CUBIC if k["cubic"] else L.WC_EOS_LINEAR
    p.wall_density = p.wall_force = int(k["wall"])
    p.mouse_force = int(k["mouse"])
    for a in range(3):
        p.gravity[a], p.camera_position[a], p.mouse_ray_direction[a] = k["g"][a], k["cam"][a], k["dir"][a]
    return L.derive(p), k


def _weights(seed):
    """Glorot-uniform parameters as one flat vector; padded rows and columns zero."""
    rng = np.random.default_rng(seed)
    out = []
    for s in SHAPES:
        w = np.zeros(s, np.float32)
        if len(s) == 2:
            r, c = min(s[0], NIN), NOUT if s[1] == NOPAD else s[1]
            a = math.sqrt(6.0 / (r + c))
            w[:r, :c] = rng.uniform(-a, a, (r, c))
        out.append(w.reshape(-1))
    return np.concatenate(out)


def _samples(rows, seed):
    """Closure inputs and targets of `rows` particles: 24 to 32 neighbours inside the unit ball, their
    velocity differences, then the three scalars."""
    gen, d = _gen(seed), _device()
    x = torch.zeros(rows, NPAD, device=d)
    nb = torch.randn(rows, 32, 6, generator=gen, device=d)
    nb[:, :, :3] *= (torch.rand(rows, 32, 1, generator=gen, device=d).pow(1 / 3) /
                     nb[:, :, :3].norm(dim=2, keepdim=True).clamp_min(1e-3))
    nb[:, :, 3:] *= 0.1
    cnt = torch.randint(24, 33, (rows, 1), generator=gen, device=d)
    nb *= (torch.arange(32, device=d)[None] < cnt)[:, :, None]
    x[:, :192] = nb.reshape(rows, 192)
    x[:, 192] = torch.randn(rows, generator=gen, device=d) * 0.3
    x[:, 193] = 1.0
    x[:, 194] = cnt[:, 0] / 32.0
    t = torch.zeros(rows, 4, device=d)
    t[:, :3] = torch.randn(rows, 3, generator=gen, device=d) * 0.2 + 0.3 * nb[:, :3, 3].sum(1, keepdim=True)
    return x.to(torch.bfloat16), t


# ---------------------------------------------------------------------------------------------
# states and passes
# ---------------------------------------------------------------------------------------------
class _Shared:
    """A device array of the package as a tensor (its owner lives as long as the tensor)."""

    def __init__(self, ptr, rows, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (rows, 4), "typestr": "<f4", "data": (int(ptr), False), "version": 2}


def _tensor(ptr, rows, owner):
    return torch.as_tensor(_Shared(ptr, rows, owner), device="cuda")


def _buffer1(owner):
    """Buffer 1 of a context: its two halves as tensors."""
    from watercube_amd import _lib as L

    v = L.wc_device_view()
    L.check(L.lib().wc_device_view_get(owner.ctx, C.byref(v)), "wc_device_view_get")
    return [_tensor(v.posrho[0], v.num_particles, owner), _tensor(v.velp[0], v.num_particles, owner)]


def prepare(case, seed):
    from watercube_amd import Fluid, batch, closure
    from watercube_amd import _lib as L

    kind = case["kind"]
    state = {"case": case}
    if kind in ("fluid", "closure_run", "closure_infer"):
        rec = _records(case, seed)
        p, k = _params(case, len(rec))
        f = Fluid(p, _numpy_records(rec)).setup()
        state.update(fluid=f, dt=k["dt"], out=_buffer1(f))
        if kind == "fluid":
            if case["tune"]:
                f.tune(k["dt"], reps=2)
            return state
        f.set_tuning(4, 8, 1)  # neighbour lists, as the tuner picks for these scenes
        state["net"] = closure.ClosureNet(max_batch=1024).load(WEIGHTS)
        if kind == "closure_infer":
            f.sort_.run()
            f.runDensityProg()
            y = torch.zeros(len(rec), 4, device="cuda")
            torch.cuda.synchronize()
            state.update(y=y, ptr=C.c_void_p(y.data_ptr()))
        return state
    if kind == "batch":
        scenes = []
        for c, sd in _batch_scenes(case, seed):
            rec = _records(c, sd)
            p, k = _params(c, len(rec))
            scenes.append((p, _numpy_records(rec), k["dt"], "block"))
        b = batch.SceneBatch(scenes).setup()
        if case["tune"]:
            b.tune(reps=2)
        state.update(batch=b, out=_buffer1(b))
        return state
    if kind == "noalloc":
        rec = _records(case, seed)
        p, k = _params(case, len(rec))
        pr, vp = rec[:, :4].contiguous(), rec[:, 4:].contiguous()
        state.update(p=p, dt=C.c_float(k["dt"]), out=[pr, vp], args=(C.c_void_p(pr.data_ptr()), C.c_void_p(vp.data_ptr())))
        return state
    rows, batches = case["rows"], case.get("batches", 1)
    x, t = _samples(rows * batches, seed)
    net = closure.ClosureNet(max_batch=rows)
    net.set_params(_weights(seed))
    xd = closure.DeviceArray((rows * batches, closure.NFEAT), np.uint16).upload(x.view(torch.int16).cpu().numpy().view(np.uint16))
    td = closure.DeviceArray((rows * batches, 4), np.float32).upload(t.cpu().numpy())
    state.update(net=net, x=xd, t=td)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "fluid":
        state["fluid"].step(state["dt"], case["steps"])
        return state["out"]
    if kind == "batch":
        state["batch"].step(1)
        return state["out"]
    from watercube_amd import _lib as L

    if kind == "noalloc":
        L.check(L.lib().wc_step_noalloc(C.byref(state["p"]), state["dt"], *state["args"], None, None), "wc_step_noalloc")
        return state["out"]
    if kind == "closure_run":
        f = state["fluid"]
        L.check(L.lib().wc_closure_set_smoothing(f.ctx, int(case["smooth"])), "wc_closure_set_smoothing")
        st = L.wc_closure_stats()
        L.check(L.lib().wc_closure_run(f.ctx, state["net"].h, C.c_float(state["dt"] / 2), case["K"], case["macro"],
                                       C.c_float(0.01), C.byref(st)), "wc_closure_run")
        return {"state": state["out"], "steps": [st.macro_steps, st.fallbacks],
                "density": [st.max_density_jump, st.peak_density]}
    if kind == "closure_infer":
        L.check(L.lib().wc_closure_infer(state["fluid"].ctx, state["net"].h, C.c_float(case["K"]), state["ptr"]),
                "wc_closure_infer")
        return state["y"]
    net, rows = state["net"], case["rows"]
    if kind == "train":
        for b in range(case["batches"]):
            net.train_step(state["x"].offset(b * rows), state["t"].offset(b * rows), rows, 1e-3)
        return net.params()
    grad, loss = net.gradient(state["x"], state["t"], rows)
    return {"gradient": grad, "loss": loss}


# ---------------------------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------------------------
def _count(case):
    return case["nx"] * case["ny"] * case["nz"] + case.get("ball", 0)


def _step_work(n, ratio):
    """Records read and written once; per accepted neighbour a distance and kernel of the density sum
    and the distance, pressure and viscosity terms of the forces."""
    pairs = n * (4 / 3 * math.pi * ratio ** 3 - 1)
    return 64.0 * n, pairs * (14 + 52)


def work(case):
    kind = case["kind"]
    fwd = 2.0 * (NIN * NH + 2 * NH * NH + NH * NOUT)
    if kind in ("fluid", "noalloc"):
        b, f = _step_work(_count(case), case["ratio"])
        return {"bytes": b * case.get("steps", 1), "flops": f * case.get("steps", 1)}
    if kind == "batch":
        each = [_step_work(_count(c), c["ratio"]) for c, _ in _batch_scenes(case, 0)]
        return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}
    if kind == "closure_run":
        n = _count(case)
        b, f = _step_work(n, case["ratio"])
        return {"bytes": (b + 16.0 * n) * case["macro"], "flops": (f + fwd * n) * case["macro"]}
    if kind == "closure_infer":
        n = _count(case)
        return {"bytes": 48.0 * n, "flops": fwd * n}
    rows = case["rows"] * case.get("batches", 1)
    params = sum(int(np.prod(s)) for s in SHAPES)
    back = 2.0 * (NIN * NH + 2 * NH * NH + NH * NOUT + 2 * NH * NH + NH * NOUT)
    state = 4.0 * params * (7 * case["batches"] if kind == "train" else 2)
    return {"bytes": rows * (2.0 * NPAD + 16.0) + state, "flops": rows * (fwd + back)}


# ---------------------------------------------------------------------------------------------
# 64-bit restatements
# ---------------------------------------------------------------------------------------------
def _sorted(k, rec):
    """Cell of every particle (float32, as the cell is defined), the stable order, first slot and count per cell."""
    R = k["R"]
    cell = (rec[:, :3].cpu() / torch.tensor(float(k["bin"]), dtype=torch.float32)).to(rec.device)
    cell = cell.to(torch.int64).clamp_(0, R - 1)
    key = (cell[:, 2] * R + cell[:, 1]) * R + cell[:, 0]
    order = torch.argsort(key, stable=True)
    count = torch.bincount(key, minlength=R ** 3)
    return cell[order], order, torch.cumsum(count, 0) - count, count


def _neighbours(k, cell, first, count, pos):
    """For each of the 27 cells and each place in a cell: the neighbour's slot, the difference of the
    positions, the distance, and whether it is an accepted neighbour.  dx outermost, dz innermost."""
    R, n = k["R"], len(pos)
    me = torch.arange(n, device=pos.device)
    for dx in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dz in (-1, 0, 1):
                c = cell + torch.tensor([dx, dy, dz], device=pos.device)
                inside = ((c >= 0) & (c < R)).all(1)
                key = ((c[:, 2] * R + c[:, 1]) * R + c[:, 0]).clamp_(0, R ** 3 - 1)
                st, ct = first[key], torch.where(inside, count[key], 0)
                for j in range(int(ct.max())):
                    u = torch.where(j < ct, st + j, me)
                    r = pos - pos[u]
                    d = r.square().sum(1).sqrt()
                    yield u, r, d, (j < ct) & (u != me) & (d < float(k["h"]))


def _exact_step(case, seed):
    """One step in 64 bits: buffer 1 (position, density) and (velocity, pressure), in sorted order."""
    k, rec = _constants(case), _records(case, seed)
    cell, order, first, count = _sorted(k, rec)
    rec = rec[order].double()
    pos, vel = rec[:, :3].contiguous(), rec[:, 4:7].contiguous()
    h, m, size = float(k["h"]), float(k["m"]), float(k["size"])
    c6, cs, cv = 315 / (64 * math.pi * h ** 9), -45 / (math.pi * h ** 6), 45 / (math.pi * h ** 6)

    def poly(d):
        return c6 * (h * h - d * d) ** 3

    rho = torch.full_like(pos[:, 0], m * c6 * h ** 6)
    for _, _, d, ok in _neighbours(k, cell, first, count, pos):
        rho += torch.where(ok, m * poly(d), 0.0)
    x = rho / float(k["rho0"])
    p = float(k["p0"]) + float(k["k"]) * (x ** 3 - 1 if k["cubic"] else rho - float(k["rho0"]))
    dens = rho.clone()
    if k["wall"]:
        far = size - h
        for a in range(3):
            q, upper = pos[:, a], pos[:, a if a < 2 else 1]  # the z term tests y on its far side
            dens += 4 * m * torch.where(q < h, poly(q), torch.where(upper > far, poly(size - q), 0.0))
    pf, vf = torch.zeros_like(pos), torch.zeros_like(pos)
    for u, r, d, ok in _neighbours(k, cell, first, count, pos):
        pair = (p + p[u]) / (2 * dens[u])
        w = torch.where(ok & (pair > 0), m * pair * (h - d) ** 2 * cs / (d + 1e-16), 0.0)
        pf -= torch.where(w[:, None] != 0, r * w[:, None], 0.0)
        vf += (vel[u] - vel) * torch.where(ok, m / dens[u] * (h - d) * cv, 0.0)[:, None]
    ext = dens[:, None] * torch.tensor(k["g"], device=pos.device, dtype=torch.float32).double()
    if k["wall"]:
        for a in range(3):
            q = pos[:, a]
            e = torch.where(q < h, -q, torch.where(q > size - h, size - q, 0.0))
            ext[:, a] += 0.01 * (h - 3) ** 2 * (e / 3) * cs
    if k["mouse"]:
        o, v = (torch.tensor(k[w], dtype=torch.float32).double().to(pos.device) for w in ("cam", "dir"))
        t1, t2 = -o / v, (size - o) / v
        if torch.minimum(t1, t2).max() <= torch.maximum(t1, t2).min():
            to = pos - o
            d = torch.linalg.cross(v.expand_as(to), to).norm(dim=1)
            w = torch.where(d <= h, -m * p * (h - d) ** 2 * cs / (d + 1e-16) * 1e-5, 0.0)
            ext += torch.where(w[:, None] != 0, to * w[:, None], 0.0)
    dt = k["dt"]
    vel = (vel + (pf + vf * float(k["mu"]) + ext) / (dens + 1e-16)[:, None] * dt).clamp(-float(k["vmax"]), float(k["vmax"]))
    pos = pos + vel * dt
    low, high = float(k["border"]), size - float(k["border"])
    vel = torch.where((pos < low) | (pos > high), -vel * float(k["damping"]), vel)
    return [torch.cat([pos.clamp(low, high), dens[:, None]], 1), torch.cat([vel, p[:, None]], 1)]


def _matrices(flat):
    out, at = [], 0
    for s in SHAPES:
        n = int(np.prod(s))
        out.append(flat[at:at + n].reshape(s))
        at += n
    return out


def _forward(flat, x):
    """Outputs, and each layer's input and pre-activation."""
    w, kept = _matrices(flat), []
    for i in range(3):
        z = x @ w[2 * i] + w[2 * i + 1]
        kept.append((x, z))
        x = z * torch.sigmoid(z)
    return (x @ w[6] + w[7])[:, :NOUT], kept + [(x, None)]


def _gradient(flat, x, t):
    y, kept = _forward(flat, x)
    loss = (y - t[:, :NOUT]).square().mean()
    w, grads = _matrices(flat), [None] * 8
    d = torch.zeros(len(x), NOPAD, device=x.device, dtype=x.dtype)
    d[:, :NOUT] = 2 * (y - t[:, :NOUT]) / (NOUT * len(x))
    for i in (3, 2, 1, 0):
        grads[2 * i], grads[2 * i + 1] = kept[i][0].T @ d, d.sum(0)
        if i:
            z = kept[i - 1][1]
            s = torch.sigmoid(z)
            d = (d @ w[2 * i].T) * (s * (1 + z * (1 - s)))
    return torch.cat([g.reshape(-1) for g in grads]), loss


def _exact_infer(case, seed):
    k, rec = _constants(case), _records(case, seed)
    cell, order, first, count = _sorted(k, rec)
    rec = rec[order].double()
    pos, vel, h, n = rec[:, :3].contiguous(), rec[:, 4:7].contiguous(), float(k["h"]), len(rec)
    cap = 96
    near = torch.full((n, cap), float("inf"), device=pos.device, dtype=torch.float64)
    slot = torch.zeros(n, cap, device=pos.device, dtype=torch.int64)
    have = torch.zeros(n, device=pos.device, dtype=torch.int64)
    m, c6 = float(k["m"]), 315 / (64 * math.pi * h ** 9)
    rho = torch.full_like(pos[:, 0], m * c6 * h ** 6)
    for u, _, d, ok in _neighbours(k, cell, first, count, pos):
        rho += torch.where(ok, m * c6 * (h * h - d * d) ** 3, 0.0)
        i = ok.nonzero()[:, 0]
        near[i, have[i]], slot[i, have[i]] = d[i], u[i]
        have += ok
    # the 32 nearest, in the order of the walk
    pick = torch.argsort(near, dim=1, stable=True)[:, :32]
    pick = torch.where(torch.isfinite(near.gather(1, pick)), pick, cap).sort(1).values
    there = pick < cap
    u = slot.gather(1, pick.clamp_max(cap - 1))
    x = torch.zeros(n, NPAD, device=pos.device, dtype=torch.float64)
    x[:, :192] = (torch.cat([(pos[u] - pos[:, None]) / h, vel[u] - vel[:, None]], 2) * there[:, :, None]).reshape(n, 192)
    x[:, 192] = 10 * (rho / float(k["rho0"]) - 1)
    x[:, 193] = case["K"] / 4
    x[:, 194] = there.sum(1) / 32
    flat = torch.from_numpy(np.load(WEIGHTS, allow_pickle=False)).double().to(pos.device)
    y = torch.zeros(n, 4, device=pos.device, dtype=torch.float64)
    y[:, :NOUT] = _forward(flat, x)[0]
    return y


def exact(case, seed):
    kind = case["kind"]
    if kind in ("fluid", "noalloc"):
        # after a second step the order of the particles itself depends on rounding; above two million
        # particles the restatement takes too long
        return _exact_step(case, seed) if case.get("steps", 1) == 1 and _count(case) <= 2_000_000 else None
    if kind == "batch":
        each = [_exact_step(c, sd) for c, sd in _batch_scenes(case, seed)]
        return [torch.cat([e[0] for e in each]), torch.cat([e[1] for e in each])]
    if kind == "closure_run":
        return None  # several large steps: the order after the first depends on rounding
    if kind == "closure_infer":
        return _exact_infer(case, seed)
    rows, batches = case["rows"], case.get("batches", 1)
    x, t = _samples(rows * batches, seed)
    x, t = x.double(), t.double()
    flat = torch.from_numpy(_weights(seed)).double().to(x.device)
    if kind == "gradient":
        grad, loss = _gradient(flat, x, t)
        return {"gradient": grad, "loss": loss}
    m, v = torch.zeros_like(flat), torch.zeros_like(flat)
    for b in range(batches):
        g, _ = _gradient(flat, x[b * rows:(b + 1) * rows], t[b * rows:(b + 1) * rows])
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        flat = flat - 1e-3 * (m / (1 - 0.9 ** (b + 1))) / ((v / (1 - 0.999 ** (b + 1))).sqrt() + 1e-8)
    return flat

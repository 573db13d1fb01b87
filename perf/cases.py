"""The work that users of this engine have it do, as timed cases.

Four kinds of pass, all through the public binding (barnes-hut_amd/__init__.py):

  sim     `Engine.step` over a stretch of hourly steps, then `Engine.get_bodies`
          (a frame of the run): the device-resident simulation, in each form.
          warm = 1: prepare() has already taken the steps that train the cost
          model, so a pass is a stretch of a running simulation; warm = 0: a
          pass is the whole run from its upload (fresh weights, the bodies
          uploaded, the first, unsorted step, training, graph capture).
  call    upload, one force evaluation, download: the drop-in for a host loop
          that keeps its own kicks and drifts.
  static  `bh_compute_accelerations_static` on device tensors and the caller's
          stream: a serving loop that may not allocate.
  direct  `Engine.direct_sum`: the FP64 error reference on a sample of bodies.

Bodies are synthetic heliocentric systems of the engine's own populations
(main belt; belt + Kuiper belt; belt + Trojan clouds + Hildas) around the Sun
and eight planets, in AU, kg and days, drawn here on the GPU from the seed.
"""
import importlib.util
import math
import pathlib
import random
import sys

import numpy as np
import torch

ROOT = pathlib.Path(__file__).resolve().parent.parent
G = 1.48812e-34          # AU^3 kg^-1 day^-2
SUN = 1.989e30
PLANET_A = (0.39, 0.72, 1.0, 1.52, 5.2, 9.54, 19.2, 30.1)
PLANET_M = (3.30e23, 4.87e24, 5.97e24, 6.42e23, 1.90e27, 5.68e26, 8.68e25, 1.02e26)
DT = 1.0 / 24.0          # one hour
TRAIN_STEPS = 50         # steps over which the engine trains its cost model by default
EXACT_PAIRS = 2.5e11     # pair interactions that exact() spends at most


def listed():
    return [
        # one small evaluation in a serving loop: launches and latency
        {"name": "static_3k", "kind": "static", "pop": "belt", "n": 2999, "theta": 1.05, "soft2": 0.0},
        # the smallest published scenario size, bit-exact form: a simulated day, then a frame
        {"name": "plain_19k", "kind": "sim", "form": "plain", "pop": "belt", "n": 19054, "theta": 1.05, "steps": 24, "warm": 0},
        # the bit-exact form at the headline size
        {"name": "plain_300k", "kind": "sim", "form": "plain", "pop": "belt", "n": 300149, "theta": 1.05, "steps": 24, "warm": 1},
        # the precision form on a small system: too few walk groups to fill the device
        {"name": "mixed_19k", "kind": "sim", "form": "mixed", "pop": "belt", "n": 19054, "theta": 1.05, "steps": 24, "warm": 0},
        # the headline: the learned schedule in a running simulation
        {"name": "learned_300k", "kind": "sim", "form": "learned", "pop": "belt", "n": 300149, "theta": 1.05, "steps": 24, "warm": 1},
        # the same system at the accurate opening angle: long interaction lists
        {"name": "mixed_300k_theta05", "kind": "sim", "form": "mixed", "pop": "belt", "n": 300149, "theta": 0.5, "steps": 24, "warm": 1},
        # a whole run from its upload: training the cost model on the way (weights returned)
        {"name": "learned_fresh_50k", "kind": "sim", "form": "learned", "pop": "trojan", "n": 50021, "theta": 1.05, "steps": 60, "warm": 0},
        # strongly uneven walk cost: Trojan clouds
        {"name": "learned_1m_trojan", "kind": "sim", "form": "learned", "pop": "trojan", "n": 1048576, "theta": 1.05, "steps": 24, "warm": 1},
        # the largest single system
        {"name": "mixed_4m_kuiper", "kind": "sim", "form": "mixed", "pop": "kuiper", "n": 4194304, "theta": 0.7, "steps": 48, "warm": 1},
        # many systems of uneven size in one step
        {"name": "ensemble_64", "kind": "sim", "form": "mixed", "pop": "belt", "systems": 64, "nmin": 10000, "nmax": 200000,
         "sizes": 0, "theta": 1.05, "steps": 48, "warm": 1},
        # the drop-in for a host loop: upload, evaluate, download
        {"name": "call_plain_19k", "kind": "call", "form": "plain", "pop": "belt", "n": 19054, "theta": 1.05, "soft2": 0.0},
        # the error check of a mixed run: the reference sum for 4,096 sampled bodies
        {"name": "direct_4096_of_300k", "kind": "direct", "pop": "belt", "n": 300149, "m": 4096, "soft2": 0.0},
    ]


def _log_size(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["sim", "sim", "sim", "sim", "ensemble", "call", "static", "direct"])
    pop = rng.choice(["belt", "kuiper", "trojan"])
    theta = rng.choice([0.5, 0.7, 1.05, 1.05, round(rng.uniform(0.4, 1.2), 3)])
    soft2 = rng.choice([0.0, 0.0, 1e-8])
    if kind == "sim":
        form = rng.choice(["plain", "mixed", "learned"])
        warm = rng.choice([0, 1, 1])
        n = _log_size(rng, 1000, 300000 if form == "plain" else 1500000)
        steps = TRAIN_STEPS + rng.randint(6, 24) if form == "learned" and not warm else rng.randint(12, 48)
        return {"kind": "sim", "form": form, "pop": pop, "n": n, "theta": theta, "steps": steps, "warm": warm}
    if kind == "ensemble":
        nmin = _log_size(rng, 1000, 20000)
        return {"kind": "sim", "form": rng.choice(["mixed", "learned"]), "pop": pop, "systems": rng.randint(2, 64),
                "nmin": nmin, "nmax": _log_size(rng, nmin, 100000), "sizes": rng.randrange(1 << 20), "theta": theta,
                "steps": rng.randint(12, 48), "warm": 1}
    if kind == "call":
        return {"kind": "call", "form": rng.choice(["plain", "plain", "mixed"]), "pop": pop,
                "n": _log_size(rng, 1000, 400000), "theta": theta, "soft2": soft2}
    if kind == "static":
        return {"kind": "static", "pop": pop, "n": _log_size(rng, 300, 65536), "theta": theta, "soft2": soft2}
    return {"kind": "direct", "pop": pop, "n": _log_size(rng, 10000, 1000000), "m": _log_size(rng, 64, 8192), "soft2": soft2}


# ------------------------------------------------------------------ inputs
def _sizes(case):
    """Bodies of each system of the case."""
    if "systems" not in case:
        return [case["n"]]
    rng = random.Random(1000003 * case["sizes"] + case["systems"])
    return [_log_size(rng, case["nmin"], case["nmax"]) for _ in range(case["systems"])]


def _orbits(count, gen, dev, amin, amax, emax, isig):
    """count Kepler orbits: positions and velocities (count, 3) about the Sun."""
    def u(lo, hi):
        return lo + (hi - lo) * torch.rand(count, generator=gen, device=dev, dtype=torch.float64)

    a, e = u(amin, amax), u(0.0, emax)
    inc = isig * torch.sqrt(-2.0 * torch.log1p(-u(0.0, 1.0)))
    node, peri, anom = (u(0.0, 2.0 * math.pi) for _ in range(3))
    ecc = anom.clone()
    for _ in range(12):
        ecc = ecc - (ecc - e * torch.sin(ecc) - anom) / (1.0 - e * torch.cos(ecc))
    root = torch.sqrt(1.0 - e * e)
    x, y = a * (torch.cos(ecc) - e), a * root * torch.sin(ecc)
    h = torch.sqrt(G * SUN * a) / (a * (1.0 - e * torch.cos(ecc)))
    vx, vy = -h * torch.sin(ecc), h * root * torch.cos(ecc)
    co, so, ci, si, cw, sw = (f(t) for t in (node, inc, peri) for f in (torch.cos, torch.sin))
    p = torch.stack([co * cw - so * sw * ci, so * cw + co * sw * ci, sw * si], 1)
    q = torch.stack([-co * sw - so * cw * ci, -so * sw + co * cw * ci, cw * si], 1)
    return p * x[:, None] + q * y[:, None], p * vx[:, None] + q * vy[:, None]


def _system(pop, n, gen, dev):
    """Sun, planets and asteroids: positions (n, 3), velocities (n, 3), masses (n)."""
    mu = G * SUN
    phase = 2.0 * math.pi * torch.rand(8, generator=gen, device=dev, dtype=torch.float64)
    a = torch.tensor(PLANET_A, device=dev, dtype=torch.float64)
    zero = torch.zeros(8, device=dev, dtype=torch.float64)
    c, s, v = torch.cos(phase), torch.sin(phase), torch.sqrt(mu / a)
    pos = [torch.zeros(1, 3, device=dev, dtype=torch.float64), torch.stack([a * c, a * s, zero], 1)]
    vel = [torch.zeros(1, 3, device=dev, dtype=torch.float64), torch.stack([-v * s, v * c, zero], 1)]
    rest = n - 9
    kuiper = rest * 3 // 10 if pop == "kuiper" else 0
    trojan = rest * 15 // 100 if pop == "trojan" else 0
    hilda = rest // 10 if pop == "trojan" else 0
    deg = math.pi / 180.0
    for count, orbit in ((rest - kuiper - 2 * trojan - hilda, (2.1, 3.3, 0.3, 5 * deg)), (kuiper, (30.0, 50.0, 0.2, 10 * deg)),
                         (hilda, (3.7, 4.2, 0.3, 5 * deg))):
        if count:
            p, w = _orbits(count, gen, dev, *orbit)
            pos.append(p)
            vel.append(w)
    for side in (60.0 * deg, -60.0 * deg):
        if trojan:
            centre = PLANET_A[4] * torch.stack([torch.cos(phase[4] + side), torch.sin(phase[4] + side), zero[0]])
            p = centre + 0.15 * torch.randn(trojan, 3, generator=gen, device=dev, dtype=torch.float64)
            r = torch.sqrt(p[:, 0] ** 2 + p[:, 1] ** 2)
            vc = torch.sqrt(mu / r)
            pos.append(p)
            vel.append(torch.stack([-vc * p[:, 1] / r, vc * p[:, 0] / r, torch.zeros_like(r)], 1))
    light = torch.exp(math.log(1e12) + (math.log(1e20) - math.log(1e12)) * torch.rand(rest, generator=gen, device=dev, dtype=torch.float64))
    mass = torch.cat([torch.tensor([SUN, *PLANET_M], device=dev, dtype=torch.float64), light])
    return torch.cat(pos), torch.cat(vel), mass


def _bodies(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    return tuple(torch.cat(parts) for parts in zip(*[_system(case["pop"], n, gen, dev) for n in _sizes(case)]))


def _sample(case, seed):
    return np.random.default_rng(seed).choice(case["n"], size=min(case["m"], case["n"]), replace=False).astype(np.int64)


# ------------------------------------------------------------------ passes
def _package():
    name = "bh_amd"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(name, ROOT / "barnes-hut_amd" / "__init__.py", submodule_search_locations=[])
        sys.modules[name] = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(sys.modules[name])
    return sys.modules[name]


def prepare(case, seed):
    bh = _package()
    pos, vel, mass = _bodies(case, seed)
    if case["kind"] == "static":
        return {"case": case, "lib": bh.load(), "pos": pos, "mass": mass, "acc": torch.empty_like(pos)}
    state = {"case": case, "host": tuple(t.cpu().numpy() for t in (pos, vel, mass)), "sizes": _sizes(case)}
    if case["kind"] == "direct":
        state["engine"] = bh.Engine()
        state["idx"] = _sample(case, seed)
        _upload(state)
        return state
    form = {"plain": bh.FORM_PLAIN, "mixed": bh.FORM_MIXED, "learned": bh.FORM_LEARNED}[case["form"]]
    state["form"] = form
    state["engine"] = bh.Engine(form=form, theta=case["theta"], soft2=case.get("soft2", 0.0))
    if case["kind"] == "sim" and case["warm"]:
        _upload(state)
        state["engine"].step(_warm_steps(case), DT)
    return state


def _warm_steps(case):
    return TRAIN_STEPS + 2 if case["form"] == "learned" else 2


def _upload(state):
    state["engine"].set_bodies(*state["host"])
    if len(state["sizes"]) > 1:
        state["engine"].set_systems(state["sizes"])


def run(state):
    case = state["case"]
    if case["kind"] == "static":
        lib, pos, acc = state["lib"], state["pos"], state["acc"]
        rc = lib.bh_compute_accelerations_static(pos.shape[0], pos.data_ptr(), state["mass"].data_ptr(), case["theta"], G, case["soft2"],
                                                 acc.data_ptr(), torch.cuda.current_stream().cuda_stream)
        if rc:
            raise RuntimeError(lib.bh_static_last_error().decode())
        return acc
    engine = state["engine"]
    if case["kind"] == "direct":
        return engine.direct_sum(state["idx"], soft2=case["soft2"])
    if case["kind"] == "call":
        _upload(state)
        engine.compute_accelerations(state["form"], case["theta"], G, case["soft2"])
        return engine.get_bodies()
    if not case["warm"]:
        if case["form"] == "learned":
            engine.model_reset(7)
        _upload(state)
    engine.step(case["steps"], DT)
    out = engine.get_bodies()
    if case["form"] == "learned" and not case["warm"]:
        out["weights"] = engine.model_get_params()
    return out


# -------------------------------------------------- the same in 64 bits, plainly
def _direct(pos, mass, soft2, at=None):
    """Accelerations of the bodies `at` (all of them: None) by direct summation."""
    at = torch.arange(pos.shape[0], device=pos.device) if at is None else at
    out = torch.empty(at.shape[0], 3, device=pos.device, dtype=torch.float64)
    rows = max(1, (1 << 26) // pos.shape[0])
    for lo in range(0, at.shape[0], rows):
        p = pos[at[lo:lo + rows]]
        d = [pos[None, :, k] - p[:, k, None] for k in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        s = torch.where(r2 > 0.0, (G * mass)[None, :] / ((r2 + soft2) * torch.sqrt(r2 + soft2)), 0.0)
        for k in range(3):
            out[lo:lo + rows, k] = (s * d[k]).sum(1)
    return out


def _morton_order(pos):
    """Order of the bodies by the 63-bit Morton key of their position in their box."""
    lo, hi = pos.min(0).values, pos.max(0).values
    span = torch.where(hi > lo, hi - lo, 1.0)
    cell = ((pos - lo) / span * (1 << 21)).to(torch.int64).clamp(0, (1 << 21) - 1)
    key = torch.zeros(pos.shape[0], device=pos.device, dtype=torch.int64)
    for bit in range(21):
        for k in range(3):
            key |= ((cell[:, k] >> bit) & 1) << (3 * bit + k)
    return torch.argsort(key, stable=True)


def exact(case, seed):
    sizes = _sizes(case)
    steps = 1 if case["kind"] != "sim" else case["steps"] + (_warm_steps(case) if case["warm"] else 0)
    pairs = steps * sum(float(n) * n for n in sizes)
    if case["kind"] == "direct":
        pairs = float(case["m"]) * case["n"]
    if pairs > EXACT_PAIRS:
        return None
    pos, vel, mass = _bodies(case, seed)
    soft2 = case.get("soft2", 0.0)
    if case["kind"] == "static":
        return _direct(pos, mass, soft2).cpu()
    if case["kind"] == "direct":
        return _direct(pos, mass, soft2, torch.from_numpy(_sample(case, seed)).to(pos.device)).cpu().numpy()
    offs = np.concatenate([[0], np.cumsum(sizes)])
    parts = [slice(int(a), int(b)) for a, b in zip(offs[:-1], offs[1:])]
    acc = torch.zeros_like(pos)
    for step in range(steps):
        if case["kind"] == "sim":
            if step:
                vel = vel + 0.5 * DT * acc
            pos = pos + DT * vel
        acc = torch.cat([_direct(pos[p], mass[p], soft2) for p in parts])
        if case["kind"] == "sim":
            vel = vel + 0.5 * DT * acc
    order = torch.cat([p.start + _morton_order(pos[p]) for p in parts])
    out = {k: v[order].cpu().numpy() for k, v in (("pos", pos), ("vel", vel), ("mass", mass), ("acc", acc))}
    out["ids"] = None
    if case["kind"] == "sim" and case["form"] == "learned" and not case["warm"]:
        out["weights"] = None
    return out


# ------------------------------------------------------------------ floors
def _accepted(n, theta):
    """Interactions per body of the opening criterion, roughly: 1,130 at 300k bodies and theta 1.05, growing with the depth of the tree."""
    return min(float(n), 215.0 * max(1.0, math.log(max(n, 64) / 64.0, 8.0)) * max(0.3, min(theta, 1.5) / 1.05) ** -2.3 * 1.3)


def work(case):
    """Bytes: each body's state read and written once a pass (and, for a host pass, moved over the bus); operations: 21 for an
    accepted interaction and 9 for a test that opens a node, about one in five, or 20 a pair of a direct sum."""
    sizes = _sizes(case)
    n = float(sum(sizes))
    if case["kind"] == "direct":
        return {"bytes": 32.0 * n + 32.0 * case["m"], "flops": 20.0 * case["m"] * n}
    flops = sum(k * _accepted(k, case["theta"]) * (21.0 + 1.8) for k in sizes)
    if case["kind"] == "static":
        return {"bytes": 56.0 * n, "flops": flops}
    if case["kind"] == "call":
        return {"bytes": (56.0 + 88.0) * n, "flops": flops}
    upload = 0.0 if case["warm"] else 56.0 * n
    return {"bytes": upload + 88.0 * n + 152.0 * n * case["steps"], "flops": flops * case["steps"]}

"""The work that programs have this framework do, as cases for timing.

Five kinds of call, each through the package's public entry points:

  run    a deck's text to results: Sim(deck), main-loop steps, the fields (the way a deck is run:
         set-up, a stretch of steps or the whole run, output)
  batch  the same for several decks that advance together in one Sim
  seam   the two per-step calls on a device-resident domain, between an upload of the state and a
         download, as a driver does that keeps its own loop
  easm   the EASM temperature on such a domain, then UpdateVoxels on it
  heat   the differentiable temperature field: loss (FP32, FP64), loss and adjoint gradient, and
         the batched gradient of a calibration step

Sizes, process parameters and melt-pool shapes are those of the decks in decks/ and of the
benchmark's workloads, or lie between them.  The seed moves the beam speed, the melt-pool
semi-axes, the grain densities and the parameter sets by a few per cent.
"""
import math
import random

import numpy as np
import torch

import amcafe_amd
from amcafe_amd.heat import HeatBatch, HeatField, track_desc

DX = 2.5e-6
TL, T0 = 1733.0, 300.0
AVEL, NVEL = 2e-5, 3.0
# melt pools (front, tail, half-width, depth in um, beam speed in m/s, power in W)
POOLS = {
    "small": (20.0, 60.0, 15.0, 12.0, 0.8, 200.0),
    "track": (64.0, 306.0, 87.0, 33.0, 0.8, 200.0),
    "batch": (46.0, 199.0, 69.0, 18.0, 1.316, 161.5),
    "raster": (67.0, 380.0, 90.0, 32.0, 1.0, 250.0),
}
# parameter sets of the heat field: power, speed, absorptivity, radius
TARGET = (220.0, 0.9, 0.4, 45e-6)
START = (200.0, 0.8, 0.35, 50e-6)


def listed():
    return [
        # one call of each seam on the smallest odd-sized domain (37x29x20): the price of a call
        {"name": "seam_small", "kind": "seam", "nx": 37, "ny": 29, "nz": 20, "pool": "small", "steps": 1, "warm": 60},
        # a driver that keeps its own loop: 32 steps on the single-track domain between transfers
        {"name": "seam_track", "kind": "seam", "nx": 128, "ny": 64, "nz": 32, "pool": "track", "steps": 32, "warm": 80},
        # the small two-layer raster, deck to result (layer change, renumbering, three tracks)
        {"name": "run_small", "kind": "run", "nx": 40, "ny": 24, "nz": 20, "pool": "small", "plate": 4, "layer": 8,
         "layers": 2, "tracks": 3, "hatch": 30.0, "grains": 200, "nuc": 1e-3, "steps": 0},
        # the single-track workload, deck to result
        {"name": "run_track", "kind": "run", "nx": 128, "ny": 64, "nz": 32, "pool": "track", "plate": 8, "layer": 24,
         "layers": 1, "tracks": 1, "hatch": 60.0, "grains": 200, "nuc": 1e-4, "steps": 0},
        # a mid-sized raster in its first track (the melt pool at its full size for most steps)
        {"name": "run_mid", "kind": "run", "nx": 256, "ny": 192, "nz": 64, "pool": "raster", "plate": 28, "layer": 12,
         "layers": 3, "tracks": 3, "hatch": 60.0, "grains": 600, "nuc": 1e-4, "steps": 300},
        # the 512x512x128 raster from its deck through its first steps
        {"name": "run_raster", "kind": "run", "nx": 512, "ny": 512, "nz": 128, "pool": "raster", "plate": 80,
         "layer": 12, "layers": 4, "tracks": 3, "hatch": 60.0, "grains": 2000, "nuc": 1e-4, "steps": 400},
        # a batch of independent single-track decks in one Sim, first steps and every deck's fields
        {"name": "batch_12", "kind": "batch", "decks": 12, "pool": "batch", "steps": 160, "nlo": 64, "nhi": 160},
        # the EASM temperature driving UpdateVoxels
        {"name": "easm_track", "kind": "easm", "nx": 128, "ny": 64, "nz": 32, "pool": "track", "steps": 2, "warm": 40},
        # the field's loss over a whole track, FP32
        {"name": "heat_forward", "kind": "heat", "what": "loss", "nx": 256, "ny": 256, "nz": 64, "steps": 2000, "sets": 1},
        # its loss and adjoint gradient
        {"name": "heat_gradient", "kind": "heat", "what": "grad", "nx": 256, "ny": 256, "nz": 64, "steps": 2000, "sets": 1},
        # one iteration of a calibration: 32 parameter sets, each against its own target
        {"name": "heat_calibration", "kind": "heat", "what": "grad", "nx": 128, "ny": 128, "nz": 48, "steps": 400, "sets": 32},
        # the FP64 loss that finite differences use, odd sizes
        {"name": "heat_f64", "kind": "heat", "what": "loss64", "nx": 125, "ny": 99, "nz": 41, "steps": 200, "sets": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run", "run", "batch", "seam", "easm", "heat", "heat"])
    if kind == "run":
        big = rng.random() < 0.5
        pool = rng.choice(["track", "raster", "batch"]) if big else "small"
        nx, ny = (_log(rng, 96, 384), _log(rng, 64, 320)) if big else (_log(rng, 24, 96), _log(rng, 20, 64))
        nz = rng.randint(40, 96) if big else rng.randint(20, 40)
        layer = rng.randint(8, 12) if big else 8
        layers = rng.randint(1, 2)
        return {"kind": "run", "nx": nx, "ny": ny, "nz": nz, "pool": pool, "plate": nz - layer * layers, "layer": layer,
                "layers": layers, "tracks": rng.randint(1, 3), "hatch": 60.0 if big else 30.0,
                "grains": _log(rng, 100, 1500), "nuc": 10.0 ** rng.uniform(-5, -3), "steps": _log(rng, 64, 280)}
    if kind == "batch":
        return {"kind": "batch", "decks": rng.randint(2, 12), "pool": "batch", "steps": rng.randint(64, 160),
                "nlo": rng.randint(40, 64), "nhi": rng.randint(80, 160)}
    if kind == "seam":
        pool = rng.choice(["small", "track"])
        return {"kind": "seam", "nx": _log(rng, 24, 200), "ny": _log(rng, 20, 96), "nz": rng.randint(18, 48), "pool": pool,
                "steps": _log(rng, 1, 40), "warm": rng.randint(30, 80)}
    if kind == "easm":
        return {"kind": "easm", "nx": _log(rng, 32, 128), "ny": _log(rng, 24, 72), "nz": rng.randint(18, 32), "pool": "track",
                "steps": rng.randint(1, 3), "warm": rng.randint(20, 50)}
    what = rng.choice(["loss", "grad", "grad", "loss64"])
    sets = _log(rng, 1, 32) if what == "grad" else 1
    hi = 256 if what != "loss64" else 120
    return {"kind": "heat", "what": what, "nx": _log(rng, 32, hi), "ny": _log(rng, 24, min(hi, 200)), "nz": rng.randint(8, 48),
            "steps": _log(rng, 20, 400), "sets": sets}


# ------------------------------------------------------------------------------------------
def _rng(case, seed):
    return random.Random("%d %s" % (seed, sorted((k, v) for k, v in case.items() if k != "name")))


def _pool(case, r):
    front, tail, half, depth, v, power = POOLS[case["pool"]]
    j = lambda x: x * r.uniform(0.96, 1.04)
    return j(front) * 1e-6, j(tail) * 1e-6, j(half) * 1e-6, j(depth) * 1e-6, j(v), power


def _solidus(v):
    return TL - (0.5 * v / AVEL) ** (1.0 / NVEL)  # half a voxel of growth a step at the most


def _deck(case, r):
    front, tail, half, depth, v, power = _pool(case, r)
    nx, ny, plate = case["nx"], case["ny"], case["plate"]
    mu = case["grains"] * r.uniform(0.9, 1.1) / (nx * 2.5 * ny * 2.5 * plate * 2.5)
    hatch = case["hatch"] * 1e-6
    if case["steps"]:  # the first steps of a longer run: the laser enters at once
        over = 0.25 * front
    else:              # a whole run: each layer's last melt pool leaves the domain
        over = hatch / 2 + tail + 12e-6
    # layers of several tracks are turned by 90 degrees: the grid spans the longer side then
    turned = case["tracks"] > 1
    length = (max(nx, ny) if turned else nx) * DX + 2 * over
    return "\n".join([
        "dx 2.5e-6", f"nX {nx} {ny} {case['nz']}", f"bmV {v!r}", f"bmP {power!r}", f"bmDelT {DX / v!r}",
        f"r {case['nuc'] * r.uniform(0.9, 1.1)!r}", f"lT {case['layer'] * DX!r}", "tL 1733", f"tS {_solidus(v)!r}",
        f"bhatch {hatch!r}", f"mu {mu!r}", f"bpH {plate * DX!r}", f"lrate {mu!r}",
        f"meltparam {front!r} {tail!r} {half!r} {depth!r}", f"patternID {2 if turned else 1}", "outint 1000000", "outNL 1",
        "offset 0.0 0.0 0.0", f"gridsize {length!r} {(case['tracks'] - 1) * hatch!r}",
        f"gridtheta {math.pi / 2 if turned else 0.0!r}", "dendritegrowth2 2e-5 3", ""])


def _batch_decks(case, r):
    decks = []
    size = _rng(case, 0)  # the decks' sizes belong to the case, their processes to the seed
    for _ in range(case["decks"]):
        nz = size.randint(40, 72)
        c = {"nx": _log(size, case["nlo"], case["nhi"]), "ny": _log(size, case["nlo"], max(case["nlo"] + 1, case["nhi"] // 2)),
             "nz": nz, "pool": case["pool"], "plate": nz - 12, "layer": 12, "layers": 1, "tracks": 1, "hatch": 60.0,
             "grains": 200, "nuc": 10.0 ** r.uniform(-5, -3), "steps": case["steps"]}
        decks.append(_deck(c, r))
    return decks


def _domain_state(case, r):
    """A domain for the seams and the state that a run of the same deck reaches after `warm` steps."""
    small = case["pool"] == "small"
    layer = 8 if small else 12
    c = {"nx": case["nx"], "ny": case["ny"], "nz": case["nz"], "pool": case["pool"], "plate": case["nz"] - layer - 2,
         "layer": layer, "layers": 1, "tracks": 1, "hatch": 30.0 if small else 60.0, "grains": 200, "nuc": 1e-4, "steps": 1}
    front, tail, half, depth, v, power = _pool(c, random.Random(r.randint(0, 1 << 30)))
    c["nuc"] *= r.uniform(0.9, 1.1)
    text = _deck(c, r)
    sim = amcafe_amd.Sim(text)
    warm = max(1, min(case["warm"], case["nx"] // 2))
    for _ in range(warm):
        sim.step()
    f = sim.fields(0, which=("gID", "vState", "extents", "centroidOct", "BuildjID"))
    grains = sim.grains(0)
    info = sim.info()
    sim.close()
    dom = amcafe_amd.Domain((case["nx"], case["ny"], case["nz"]), DX, TL, _solidus(v), T0, (front, tail, half, depth), v,
                            DX / v, c["nuc"], AVEL, NVEL)
    return {"dom": dom, "fields": f, "grains": grains, "il": info["ilaserLoc"], "t0": info["tInd"],
            "x0": warm * DX, "y": 0.5 * case["ny"] * DX, "power": power, "layerT": layer * DX}


def _heat_sets(case, r):
    near = lambda p, s: [x * r.uniform(1 - s, 1 + s) for x in p]
    return [near(TARGET, 0.1) for _ in range(case["sets"])], [near(START, 0.05) for _ in range(case["sets"])]


def prepare(case, seed):
    r = _rng(case, seed)
    kind = case["kind"]
    if kind == "run":
        return {"case": case, "decks": [_deck(case, r)]}
    if kind == "batch":
        return {"case": case, "decks": _batch_decks(case, r)}
    if kind in ("seam", "easm"):
        return {"case": case, **_domain_state(case, r)}
    targets, starts = _heat_sets(case, r)
    desc = track_desc((case["nx"], case["ny"], case["nz"]), steps=case["steps"])
    field = HeatField(desc, targets[0]) if case["sets"] == 1 else HeatBatch(desc, targets)
    return {"case": case, "field": field, "starts": starts}


def _run_decks(case, decks):
    sim = amcafe_amd.Sim(decks)
    n = 0
    while sim.step() > 0:
        n += 1
        if n == case["steps"]:
            break
    # the result of a batch's decks and of the largest domain is the microstructure, the others' the
    # whole state
    which = ("gID", "vState", "TempCurr", "extents", "centroidOct", "BuildjID", "Build")
    if case["kind"] == "batch":
        which = ("gID", "vState", "extents", "Build")
    elif case["nx"] * case["ny"] * case["nz"] > (1 << 23):
        which = ("gID", "vState", "Build")
    out = []
    for i in range(len(decks)):
        f = sim.fields(i, which=which)
        out.append([f[k] for k in which] + [np.array([sim.info(i)["tInd"], sim.info(i)["nGrain"], sim.stats(i)["n_events"]])])
    sim.close()
    return out


def _run_domain(s):
    case, dom = s["case"], s["dom"]
    dom.upload(**s["fields"])
    dom.set_grains(s["grains"])
    counts = []
    for k in range(case["steps"]):
        x, z = s["x0"] + k * DX, s["il"] * DX
        if case["kind"] == "easm":
            counts.append(dom.easm_temperature(x, s["y"], z, 1.0, 0.0, s["il"], s["power"], s["layerT"])[0])
        else:
            counts.append(dom.temperature(x, s["y"], z, 1.0, 0.0, s["il"]))
        st = dom.update_voxels(s["t0"] + k, s["il"])
        counts += [st["n_active"], st["n_events"], st["n_captures"], st["n_nucleations"]]
    return [dom.download(), np.array(counts)]


def run(state):
    case = state["case"]
    if case["kind"] in ("run", "batch"):
        out = _run_decks(case, state["decks"])
        return out[0] if len(out) == 1 else out
    if case["kind"] in ("seam", "easm"):
        return _run_domain(state)
    f, n = state["field"], case["steps"]
    if case["sets"] > 1:
        loss, grad, _ = f.loss_grad_f32(state["starts"], 0, n)
        return [np.array(loss, np.float32), np.array(grad, np.float32)]
    if case["what"] == "loss64":
        return np.array([f.loss_f64(state["starts"][0], 0, n)[0]])
    if case["what"] == "loss":
        return np.array([f.loss_f32(state["starts"][0], 0, n)[0]], np.float32)
    loss, grad, _ = f.loss_grad_f32(state["starts"][0], 0, n)
    return [np.array([loss], np.float32), np.array([grad], np.float32)]


def work(case):
    """Bytes and operations one pass cannot do without."""
    kind = case["kind"]
    if kind == "heat":
        # per voxel, step and quadrature node: a product and a sum for the field and one for the
        # target's (and three more sums for a gradient); about 20 operations for the two
        # indicators.  The heated band holds about a sixth of the voxel-steps (FP32 skips the rest).
        vs = case["nx"] * case["ny"] * case["nz"] * case["steps"] * case["sets"]
        share = 1.0 if case["what"] == "loss64" else 0.16
        ops = {"loss": 25 * 4 + 20, "loss64": 25 * 4 + 20, "grad": 25 * 10 + 40}[case["what"]]
        return {"bytes": 64.0 * case["sets"], "flops": vs * share * ops}
    front, tail, half, depth, _, _ = POOLS[case["pool"]]
    if kind == "batch":
        side = math.sqrt(case["nlo"] * case["nhi"])
        n, nvox = case["decks"], case["decks"] * side * side * 0.7 * 56
        nx, ny = side, 0.7 * side
    else:
        n, nx, ny, nvox = 1, case["nx"], case["ny"], case["nx"] * case["ny"] * case["nz"]
    # interface cells: the solidifying surface of the half-ellipsoid behind the beam, in voxels
    area = math.pi / 2 * min(tail / 2.5, nx) * min(half / 2.5, ny / 2) + 2 * depth / 2.5 * min(tail / 2.5, nx)
    per_cell = 26 * 8 + 60  # a cell's capture distances and its state, read and written once a step
    steps = case["steps"] or (case["nx"] * case["tracks"] * case["layers"])
    if kind in ("run", "batch"):
        large = kind == "run" and nvox > (1 << 23)
        out = 12 if large else 20 if kind == "batch" else 56
        return {"bytes": nvox * (41.0 + out) + n * steps * area * per_cell,
                "flops": n * steps * area * 26 * 30}
    nbytes = nvox * (44.0 + 52.0) + steps * area * per_cell
    if kind == "easm":  # about three source integrals of 25 nodes for a voxel and step
        return {"bytes": nbytes, "flops": nvox * steps * 3 * 25 * 40.0}
    return {"bytes": nbytes, "flops": steps * area * 26 * 30}


# ------------------------------------------------------------------------------------------
# 64-bit values of the heat field: the 25-point Gauss-Legendre sum of the moving Gaussian
# source, whose terms are products of a factor of (y, z) and one of (x, t).
def _nodes(desc):
    xi, w = np.polynomial.legendre.leggauss(25)
    h = desc.t_hist / 2
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    return torch.tensor(h * (1 - xi), device=dev), torch.tensor(h * w, device=dev), dev


def _factors(desc, theta, tau, W, dy2, dz2, cols_x, cols_t):
    P, v, eta, sigma = theta
    C = eta * P / (math.pi * (desc.k / desc.alpha) * math.sqrt(4 * math.pi * desc.alpha))
    A = 2 * desc.alpha * tau + sigma ** 2
    D1 = 2 * A
    a = W * C / (tau.sqrt() * A) * torch.exp(-dy2[:, None] / D1 - dz2[:, None] / (4 * desc.alpha * tau))
    d = cols_x[:, None] - v * (cols_t[:, None] - tau)
    g = torch.exp(-d * d / D1)
    gv = g * 2 * d * (cols_t[:, None] - tau) / D1
    gs = g * (-2 * sigma / A + 4 * sigma / (D1 * D1) * d * d)
    gy = g * (4 * sigma / (D1 * D1))
    return a, g, gv, gs, gy


def _exact_heat(desc, theta, target, steps, gradient):
    tau, W, dev = _nodes(desc)
    nx, ny, nz = desc.nX[0], desc.nX[1], desc.nX[2]
    ar = lambda n: (torch.arange(n, device=dev, dtype=torch.float64) + 0.5) * desc.dX
    x = ar(nx) - desc.x_start
    dy2 = ((ar(ny) - desc.y_track) ** 2).repeat(nz)
    dz2 = ((ar(nz) - desc.z_track) ** 2).repeat_interleave(ny)
    per = max(1, (1 << 24) // (nx * ny * nz))
    out = torch.zeros(5, device=dev, dtype=torch.float64)
    for m in range(0, steps, per):
        t = torch.arange(m + 1, min(steps, m + per) + 1, device=dev, dtype=torch.float64) * desc.dt
        cx, ct = x.repeat(len(t)), t.repeat_interleave(nx)
        a, g, gv, gs, gy = _factors(desc, theta, tau, W, dy2, dz2, cx, ct)
        b, h = _factors(desc, target, tau, W, dy2, dz2, cx, ct)[:2]
        rise = a @ g.T
        s1 = torch.sigmoid((desc.T0 + rise - desc.tL) / desc.width)
        s2 = torch.sigmoid((desc.T0 + b @ h.T - desc.tL) / desc.width)
        out[0] += ((s1 - s2) ** 2).sum()
        if gradient:
            lam = 2 * (s1 - s2) * s1 * (1 - s1) / desc.width
            out[1] += (lam * rise).sum() / theta[0]
            out[3] += (lam * rise).sum() / theta[2]
            out[2] += (lam * (a @ gv.T)).sum()
            out[4] += (lam * (a @ gs.T + dy2[:, None] * (a @ gy.T))).sum()
    return out.cpu().numpy()


# 64-bit EASM temperatures (the 316L properties of the iterate, damped Picard iteration from 0 K).
def _exact_easm(case, x, power, v, il, layerT):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    xi, w = np.polynomial.legendre.leggauss(25)
    t, sigma, eta = 80.0e-5, 50.0e-6, 0.56
    s = torch.tensor(t / 2 * (1 + xi), device=dev)
    w = torch.tensor(t / 2 * w, device=dev)
    ar = lambda n: (torch.arange(n, device=dev, dtype=torch.float64) + 0.5) * DX
    Z, Y, X = torch.meshgrid(ar(case["nz"]), ar(case["ny"]), ar(case["nx"]), indexing="ij")
    z = il * DX
    out = torch.zeros_like(X)
    ahead = (X > x) & (Z > z - layerT) & ~(Z > z)
    out[ahead] = 0.99 * T0
    solve = ~(Z > z) & ~ahead
    d2 = ((X[solve][:, None] - (x - v * t + v * s)) ** 2) + ((Y[solve] - 0.5 * case["ny"] * DX) ** 2)[:, None]
    z2 = ((Z[solve] - z) ** 2)[:, None]

    def integral(T, at):
        cold, mid = T < 1660, (T >= 1660) & (T < 3090)
        rho = torch.where(cold, 8084.2 - 0.42086 * T - 3.8942e-5 * T * T,
                          torch.where(mid, 7432.7 + 3.9338e-2 * T - 1.8007e-4 * T * T, torch.full_like(T, 6124.72)))
        cp = torch.where(cold, 458.984 + 0.1328 * T, torch.full_like(T, 769.855))
        k = torch.where(cold, 9.248 + 1.571e-2 * T, torch.where(mid, 12.41 + 3.279e-3 * T, torch.full_like(T, 21.6465)))
        alpha = k / (rho * cp)
        a4 = 4 * alpha[:, None] * (t - s)
        C = eta * power / (math.pi * rho * cp * torch.sqrt(4 * math.pi * alpha))
        f = (t - s) ** -0.5 / (a4 / 2 + sigma ** 2) * torch.exp(-d2[at] / (a4 + 2 * sigma ** 2) - z2[at] / a4)
        return 300 + C * (f * w).sum(1)

    T = torch.empty(d2.shape[0], device=dev, dtype=torch.float64)
    at = torch.arange(d2.shape[0], device=dev)
    old = torch.zeros_like(T)
    new = integral(old, at)
    for n in range(101):
        more = ((old - new).abs() > 10) & (n < 100)
        T[at[~more]] = new[~more]
        at, old = at[more], new[more]
        if not len(at):
            break
        new = 0.5 * (old + integral(old, at))
    out[solve] = T
    return out.reshape(-1).cpu().numpy()


# The other outputs follow from the state before, event by event: their whole numbers and
# positions have no plain formula.
def exact(case, seed):
    r = _rng(case, seed)
    if case["kind"] == "easm":
        v, power = _pool(case, random.Random(r.randint(0, 1 << 30)))[4:]
        small = case["pool"] == "small"
        x = max(1, min(case["warm"], case["nx"] // 2)) * DX + (case["steps"] - 1) * DX
        T = _exact_easm(case, x, power, v, case["nz"] - 2, (8 if small else 12) * DX)
        return [{"TempCurr": T}, None]
    if case["kind"] != "heat":
        return None
    targets, starts = _heat_sets(case, r)
    desc = track_desc((case["nx"], case["ny"], case["nz"]), steps=case["steps"])
    gradient = case["what"] == "grad"
    got = [_exact_heat(desc, s, t, case["steps"], gradient) for s, t in zip(starts, targets)]
    if not gradient:
        return np.array([got[0][0]])
    return [np.array([g[0] for g in got]), np.array([g[1:] for g in got])]

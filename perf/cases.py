"""The work a user of the engine has it do, as timed cases.

Five kinds of call, each through the package's public entry points:

  life     a run of photon-packet histories with peel-off to the instruments, and the images read
           back: the loop that a simulation spends its time in.  Every grid type, both
           precisions, several wavelengths and instruments, stored radiation field, guided
           scattering, batched instances; on the persistent engine, which the launch tuning
           picks for every one of them.
  tau      optical depths along a set of rays given in host memory (probes, column maps).
  paths    path segments along a set of rays that lie in device memory, into device buffers
           (callers that do their own transport on the segments).
  density  cell densities of a resident grid, sampled from the disk model: the last step of every
           set-up.
  guide    loss and parameter gradient of the path guide for a set of training records.

A case is a dict of plain values.  The grid belongs to the case; the medium on it, the rays, the
records and the random streams are made from the seed.
"""

from __future__ import annotations

import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PC = 3.08567758e16  # parsec (m)
HALF = 10 * PC      # half the side of the domain
SEXT = 1.5e-29      # extinction cross section per hydrogen atom (m2)
HR, HZ = 3 * PC, 0.3 * PC  # scale length and height of the disk

# waiting lanes per transition round that the engine's own launch tuning settles on per grid
THRESHOLD = {"cartesian": 64, "octree": 16, "voronoi": 32, "tetra": 64}


def _pkg():
    name = "skirt9_gpu_amd"
    if name in sys.modules:
        return sys.modules[name]
    home = os.path.join(ROOT, "skirt9-gpu_amd")
    spec = importlib.util.spec_from_file_location(name, os.path.join(home, "__init__.py"), submodule_search_locations=[home])
    mod = importlib.util.module_from_spec(spec)
    sys.modules[name] = mod
    spec.loader.exec_module(mod)
    return mod


def _workloads():
    _pkg()
    from skirt9_gpu_amd import workloads
    return workloads


# ------------------------------------------------------------------------------------- cases
def _life(name, grid, size, packets, tau, **more):
    case = dict(name=name, kind="life", grid=grid, size=size, packets=packets, tau=tau, nlambda=1, frames=1, pixels=200,
                precision="fp64", field=False, guided=False, instances=0)
    case.update(more)
    return case


def listed():
    return [
        # a quick look while a model is being set up: a coarse grid and a few thousand packets
        _life("cartesian_quick_look", "cartesian", 32, 4096, 1.0, pixels=100),
        # the standard benchmark disk on a regular grid, one wavelength
        _life("cartesian_disk", "cartesian", 64, 1 << 21, 1.0),
        # the production run of the benchmark: a spiral disk on a deep adaptive tree, optically
        # thick, five wavelengths
        _life("octree_thick_disk", "octree", 10, 1 << 21, 50.0, nlambda=5, frames=1),
        # a spectral cube: many wavelengths, optically thin, single precision sums
        _life("octree_cube_fp32", "octree", 9, 300_000, 1.0, nlambda=40, precision="fp32"),
        # scattering directions from the learned guide
        _life("octree_guided", "octree", 9, 1 << 18, 10.0, nlambda=5, guided=True),
        # a run that also stores the radiation field for dust heating
        _life("octree_radiation_field", "octree", 8, 200_000, 5.0, nlambda=8, field=True),
        # a clumpy medium on an unstructured mesh, seen by three instruments
        _life("voronoi_clumpy", "voronoi", 400_000, 1 << 18, 5.0, frames=3),
        # a parameter study: many small simulations on one tetrahedral mesh in one launch
        _life("tetra_parameter_study", "tetra", 150_000, 1 << 20, 1.0, instances=64, pixels=100),
        # optical depths along rays for a column map
        dict(name="octree_column_map", kind="tau", grid="octree", size=8, rays=250_000, tau=5.0, precision="fp64"),
        # path segments for a caller's own transport
        dict(name="voronoi_paths", kind="paths", grid="voronoi", size=100_000, rays=65_536),
        # cell densities of a production grid
        dict(name="octree_densities", kind="density", grid="octree", size=9, samples=100, spiral=True),
        # one gradient evaluation of the path guide on a batch of training records
        dict(name="guide_gradient", kind="guide", records=32_768),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    # kinds in the proportions of the listed cases
    kind = rng.choice(["life"] * 8 + ["tau", "paths", "density", "guide"])
    if kind == "guide":
        return dict(kind=kind, records=_log(rng, 64, 100_000))
    grid = rng.choice(["cartesian", "octree", "octree", "voronoi", "tetra"])
    size = {"cartesian": _log(rng, 16, 100), "octree": rng.choice([6, 7, 8, 9]), "voronoi": _log(rng, 5_000, 200_000),
            "tetra": _log(rng, 5_000, 100_000)}[grid]
    tau = round(math.exp(rng.uniform(math.log(0.1), math.log(50.0))), 3)
    precision = rng.choice(["fp64", "fp64", "fp32"])
    if kind == "tau":
        return dict(kind=kind, grid=grid, size=size, rays=_log(rng, 1_000, 250_000), tau=tau, precision=precision)
    if kind == "paths":
        return dict(kind=kind, grid=grid, size=size, rays=_log(rng, 500, 65_536))
    if kind == "density":
        grid = rng.choice(["cartesian", "octree", "tetra"])
        size = {"cartesian": _log(rng, 16, 100), "octree": rng.choice([6, 7, 8, 9]), "tetra": _log(rng, 5_000, 100_000)}[grid]
        return dict(kind=kind, grid=grid, size=size, samples=rng.choice([10, 33, 100]), spiral=rng.random() < 0.5)
    option = rng.choice(["none", "none", "none", "guided", "field", "instances"])
    case = _life("", grid, size, _log(rng, 1_000, 1_000_000 if grid in ("cartesian", "octree") else 200_000), tau,
                 nlambda=rng.choice([1, 1, 3, 5, 12, 40]), frames=rng.choice([1, 1, 2, 3]), pixels=_log(rng, 20, 250),
                 precision=precision)
    del case["name"]
    if option in ("guided", "field"):
        case[option] = True
    elif option == "instances":
        case["instances"] = rng.randint(2, 48)
    return case


# ----------------------------------------------------------------------- media and rays (numpy)
def _rho(x, y, z, phase):
    """The exponential disk with a two-armed spiral perturbation, relative to its centre."""
    R = np.sqrt(x * x + y * y)
    arm = np.sin(np.log((R + 1e-9 * HR) / HR) / math.tan(math.radians(15.0)) + phase - np.arctan2(y, x)) ** 2
    return np.exp(-R / HR - np.abs(z) / HZ) * (0.5 + arm)


def _tree(case, seed):
    """A density-refined octree in creation order: per node its level and integer position, the
    subdivision flags (the same for every seed), and per leaf (in node order) its density for the
    case's optical depth, with the spiral at the seed's phase."""
    phase = 2 * math.pi * np.random.default_rng(seed).random()
    maxlev, minlev = case["size"], min(4, case["size"])
    # fraction of the disk's mass above which a cell is divided: the deeper the tree, the smaller
    frac = 4.0 * 8.0 ** (-0.75 * maxlev)
    n0 = case.get("tau", 1.0) / (SEXT * 2 * HZ)  # face-on optical depth through the centre
    mass = 4 * math.pi * HR * HR * HZ
    lev, pos, flags = [], [], []
    cur = np.zeros((1, 3), np.int64)
    off = np.array([[q & 1, (q >> 1) & 1, q >> 2] for q in range(8)], np.int64)
    dens = []
    for level in range(maxlev + 1):
        h = 2 * HALF / (1 << level)
        c = (cur + 0.5) * h - HALF
        # the mean over eight points per cell, so that the thin disk is seen by coarse cells
        r, here = np.zeros(len(cur)), np.zeros(len(cur))
        for q in range(8):
            d = (off[q] - 0.5) * 0.5 * h
            at = (c[:, 0] + d[0], c[:, 1] + d[1], c[:, 2] + d[2])
            r += 0.125 * _rho(*at, 0.0)
            here += 0.125 * _rho(*at, phase)
        div = (level < minlev) | ((r * h ** 3 > frac * mass) & (level < maxlev))
        if level == maxlev:
            div[:] = False
        lev.append(np.full(len(cur), level))
        pos.append(cur)
        flags.append(div)
        dens.append(n0 * here)
        cur = (2 * cur[div][:, None, :] + off[None]).reshape(-1, 3)
        if len(cur) == 0:
            break
    lev, pos, flags, dens = (np.concatenate(v) for v in (lev, pos, flags, dens))
    return lev, pos, flags, dens[~flags]


def _borders(n):
    return np.array([-HALF + 2 * HALF * i / n for i in range(n + 1)])


def _cart_density(case, seed):
    n = case["size"]
    phase = 2 * math.pi * np.random.default_rng(seed).random()
    c = 0.5 * (_borders(n)[1:] + _borders(n)[:-1])
    X, Y, Z = np.meshgrid(c, c, c, indexing="ij")
    return (case.get("tau", 1.0) / (SEXT * 2 * HZ)) * _rho(X, Y, Z, phase).reshape(-1)


def _rays(case, seed):
    """Rays from positions in the disk and, one in ten, from outside the domain toward the disk;
    isotropic directions, one in fifty along an axis."""
    rng = np.random.default_rng(seed + 17)
    n = case["rays"]
    R, phi = rng.gamma(2.0, HR / 2, n), 2 * np.pi * rng.random(n)
    p = np.stack([R * np.cos(phi), R * np.sin(phi), rng.laplace(0, HZ, n)], axis=1)
    p = np.clip(p, -0.98 * HALF, 0.98 * HALF)
    k = rng.normal(size=(n, 3))
    k /= np.linalg.norm(k, axis=1, keepdims=True)
    axis = rng.random(n) < 0.02
    k[axis] = np.eye(3)[rng.integers(0, 3, axis.sum())] * rng.choice([-1.0, 1.0], axis.sum())[:, None]
    out = rng.random(n) < 0.1
    p[out] -= 4 * HALF * k[out]
    return np.concatenate([p, k], axis=1)


# ------------------------------------------------------------------------------------ prepare
def _upload_grid(case, seed, eng):
    """The grid and its medium, as a program uploads them."""
    pkg = _pkg()
    box = np.array([-HALF] * 3 + [HALF] * 3)
    grid = case["grid"]
    if grid == "cartesian":
        b = _borders(case["size"])
        eng.grid_cartesian(b, b, b)
        eng.medium(_cart_density(case, seed))
    elif grid == "octree":
        _, _, flags, dens = _tree(case, seed)
        tree = pkg.Octree.from_flags(box, flags)
        tree.upload(eng)
        tree.close()
        eng.medium(dens)
    else:
        # half of the points follow the disk, half fill the domain
        n = case["size"]
        pts = np.concatenate([_workloads().disk_points(n // 2, box, seed=n),
                              HALF * (2 * np.random.default_rng(n).random((n - n // 2, 3)) - 1)])
        mesh = pkg.Voronoi.build(pts, box) if grid == "voronoi" else pkg.Tetra.build(pts, box)
        mesh.upload(eng)
        cells = eng.num_cells()
        mesh.close()
        # a clumpy medium: lognormal cell densities around the mean for the optical depth
        mean = case.get("tau", 1.0) / (SEXT * 2 * HALF)
        eng.medium(mean * np.exp(np.random.default_rng(seed).normal(0.0, 1.0, cells) - 0.5))


def _prepare_life(case, seed):
    pkg, wl = _pkg(), _workloads()
    eng = pkg.Engine(0)
    nl, grid, inst = case["nlambda"], case["grid"], case["instances"]
    if grid == "octree" and case["size"] >= 10:
        # the benchmark's own set-up: refinement and cell densities on the GPU
        w = wl.octree_spiral(tau_v=case["tau"], nlambda=1, max_level=case["size"], engine=eng)
        eng.medium(w.density * np.exp(np.random.default_rng(seed).normal(0.0, 0.2, len(w.density))))
        w.octree.close()
    else:
        _upload_grid(case, seed, eng)
    lam = np.array([0.55e-6]) if nl == 1 else wl.log_wavelengths(0.3, 3.0, nl)
    sext = SEXT * (lam / 0.55e-6) ** -1.5
    eng.dust(lam, sext, np.linspace(0.6, 0.3, nl) * sext, np.linspace(0.6, 0.4, nl))
    packets = case["packets"]
    if inst:
        rng = np.random.default_rng(seed + 5)
        share = np.exp(rng.uniform(0.0, math.log(100.0), inst))
        counts = np.maximum(1, np.floor(packets * share / share.sum())).astype(np.uint64)
        packets = int(counts.sum())
        for i in range(inst):
            eng.frame_add(np.radians(rng.uniform(0, 90)), 0.0, 0.0, case["pixels"], case["pixels"], 2 * HALF, 2 * HALF)
    else:
        for f in range(case["frames"]):
            eng.frame_add(np.radians([60.0, 0.0, 90.0][f]), np.radians([0.0, 0.0, 30.0][f]), 0.0, case["pixels"], case["pixels"],
                          2 * HALF, 2 * HALF)
    eng.source_point((0.0, 0.0, 0.0), np.full(nl, 1.0 / packets))
    if inst:
        scale = np.exp(rng.uniform(math.log(0.1), math.log(20.0), inst))
        eng.instances(counts, np.arange(inst) + 1000 + seed, scale, np.repeat(1.0 / counts[:, None], nl, axis=1),
                      np.arange(inst), np.ones(inst))
    eng.options(0.5, 1e4, 0, pkg.SKG_FP64 if case["precision"] == "fp64" else pkg.SKG_FP32_KAHAN, seed + 1)
    if case["field"]:
        eng.rf_enable()
    if case["guided"]:
        eng.guide_params(_theta(seed))
        eng.guide_mode(1, 0.5, HALF)
    eng.tune(0, 256, THRESHOLD[grid])
    eng.tune_pipeline(pkg.SKG_MODE_PERSISTENT)
    return dict(case=case, eng=eng, packets=packets)


def _prepare_density(case, seed):
    pkg = _pkg()
    eng = pkg.Engine(0)
    _upload_grid(case, seed, eng)
    phase = 2 * math.pi * np.random.default_rng(seed).random()
    return dict(case=case, eng=eng, seed=seed + 3,
                model=pkg.disk_model(tau_v=5.0, sext_v=SEXT, spiral=case["spiral"], phase_zero=phase))


def _theta(seed):
    """Random parameters of the guide's network: He-scaled weights, zero biases, a small last layer."""
    rng = np.random.default_rng(seed)
    parts = []
    for nin, nout in ((9, 64), (64, 64), (64, 64), (64, 40)):
        parts += [rng.normal(0, math.sqrt(2.0 / nin), nin * nout) * (0.1 if nout == 40 else 1.0), np.zeros(nout)]
    return np.concatenate(parts).astype(np.float32)


def _records(case, seed):
    """Training records: features of scattering events in the disk, the direction taken and a
    heavy-tailed weight (the luminosity detected after the event)."""
    rng = np.random.default_rng(seed + 2)
    n = case["records"]
    R, phi = np.minimum(rng.gamma(2.0, 0.15, n), 1.0), 2 * np.pi * rng.random(n)
    p = np.stack([R * np.cos(phi), R * np.sin(phi), np.clip(rng.laplace(0, 0.03, n), -1, 1)], axis=1)

    def unit():
        k = rng.normal(size=(n, 3))
        return k / np.linalg.norm(k, axis=1, keepdims=True)

    rec = np.zeros((n, 16), np.float32)
    rec[:, 0:3] = p
    rec[:, 3:6] = unit()
    rec[:, 6] = rng.uniform(-1.0, 1.0, n)
    rec[:, 7] = np.linalg.norm(p, axis=1)
    rec[:, 8] = np.abs(p[:, 2])
    rec[:, 9:12] = unit()
    rec[:, 12] = rng.lognormal(0.0, 1.0, n) / n
    return rec


def prepare(case, seed):
    kind = case["kind"]
    if kind == "life":
        return _prepare_life(case, seed)
    if kind == "density":
        return _prepare_density(case, seed)
    pkg = _pkg()
    eng = pkg.Engine(0)
    if kind == "guide":
        eng.guide_params(_theta(seed))
        return dict(case=case, eng=eng, records=_records(case, seed))
    _upload_grid(case, seed, eng)
    eng.dust([0.55e-6], [SEXT], [0.6 * SEXT], [0.6])
    rays = _rays(case, seed)
    if kind == "tau":
        return dict(case=case, eng=eng, rays=rays, fp=pkg.SKG_FP64 if case["precision"] == "fp64" else pkg.SKG_FP32_KAHAN)
    # device buffers large enough for any set of such rays
    n, size = case["rays"], case["size"]
    cap = int(n * 1.3 * _crossings(case)) + 1000
    dev = torch.device("cuda", 0)
    state = dict(case=case, eng=eng, rays=torch.from_numpy(rays).to(dev), cap=cap,
                 off=torch.zeros(n + 1, dtype=torch.int64, device=dev), m=torch.zeros(cap, dtype=torch.int32, device=dev),
                 ds=torch.zeros(cap, dtype=torch.float64, device=dev))
    torch.cuda.synchronize()  # the engine reads these on its own stream
    return state


# ---------------------------------------------------------------------------------------- run
def run(state):
    case, eng = state["case"], state["eng"]
    kind = case["kind"]
    if kind == "life":
        eng.frame_clear()
        if case["field"]:
            eng.rf_clear()
        eng.run_packets(0, state["packets"])
        frames = case["instances"] or case["frames"]
        out = {"images": [eng.frame_read(f) for f in range(frames)] if frames <= 8 else
               np.stack([eng.frame_read(f) for f in range(frames)])}
        if case["field"]:
            out["field"] = eng.rf_read()
        # histories, peel-offs, forced passes, scatterings, cell crossings, second passes
        out["counters"] = eng.counters()[[0, 1, 2, 3, 4, 6]]
        return out
    if kind == "tau":
        path, obs = eng.trace_tau(state["rays"], 0, 1.0, state["fp"])
        return {"path": path, "obs": obs}
    if kind == "paths":
        total = eng.trace_paths_noalloc(state["rays"].data_ptr(), case["rays"], state["cap"], state["off"].data_ptr(),
                                        state["m"].data_ptr(), state["ds"].data_ptr())
        return {"total": total, "off": state["off"], "m": state["m"], "ds": state["ds"]}
    if kind == "density":
        return eng.sample_density(state["model"], case["samples"], state["seed"])
    grad, loss = eng.guide_gradient(state["records"])
    return {"grad": grad, "loss": loss}


# --------------------------------------------------------------------------------------- work
def _cells(case):
    g, s = case["grid"], case["size"]
    if g == "octree":
        return 11_500 * 4.38 ** (s - 6)
    return {"cartesian": s ** 3, "voronoi": s, "tetra": 6.5 * s}[g]


def _crossings(case):
    """Cells along a typical ray of _rays()."""
    g, s = case["grid"], case["size"]
    if g == "octree":
        return 25.0 * 1.53 ** (s - 6)
    return {"cartesian": 1.0 * s, "voronoi": 1.2 * s ** (1 / 3), "tetra": 3.6 * s ** (1 / 3)}[g]


# per cell crossing: the bytes of the cell's own geometry, neighbours and density, and the FP64
# operations of the exit search
CROSSING = {"cartesian": (8, 25), "octree": (112, 25), "voronoi": (500, 200), "tetra": (250, 80)}


def work(case):
    kind = case["kind"]
    if kind == "guide":
        params = 11_560
        return {"bytes": 64.0 * case["records"] + 8.0 * params, "flops": 6.0 * params * case["records"]}
    cells = _cells(case)
    if kind == "density":
        # per sample: three random numbers, two exponentials, a square root, the spiral's terms
        return {"bytes": 56.0 * cells, "flops": cells * case["samples"] * (150.0 if case["spiral"] else 80.0)}
    table, ops = CROSSING[case["grid"]]
    if kind in ("tau", "paths"):
        crossed = case["rays"] * _crossings(case)
        moved = 48.0 * case["rays"] + table * min(cells, crossed) + (16.0 * case["rays"] if kind == "tau" else 12.0 * crossed)
        return {"bytes": moved, "flops": crossed * (ops + 2)}
    # about three events per history, each with a peel-off per instrument and a forced path
    looks = 1 if case["instances"] else case["frames"]
    crossed = case["packets"] * 2.5 * (looks + 1.2) * _crossings(case)
    pixels = case["nlambda"] * (case["instances"] or case["frames"]) * float(case["pixels"]) ** 2
    moved = table * min(cells, crossed) + 8.0 * pixels + (8.0 * cells * case["nlambda"] if case["field"] else 0.0)
    return {"bytes": moved, "flops": crossed * (ops + 2)}


# -------------------------------------------------------------------------------------- exact
def _exact_tau_cartesian(case, seed):
    b, n = _borders(case["size"]), case["size"]
    dens = _cart_density(case, seed).reshape(n, n, n)
    rays = _rays(case, seed)
    tau = np.zeros(len(rays))
    for s in range(0, len(rays), 4096):
        r, k = rays[s:s + 4096, :3], rays[s:s + 4096, 3:]
        with np.errstate(divide="ignore", invalid="ignore"):
            t = np.concatenate([np.where(np.abs(k[:, a:a + 1]) > 1e-15, (b[None] - r[:, a:a + 1]) / k[:, a:a + 1], np.inf)
                                for a in range(3)], axis=1)
        t = np.sort(np.where(np.isfinite(t), np.maximum(t, 0.0), np.nan), axis=1)
        t = np.where(np.isnan(t), np.nanmax(t, axis=1, keepdims=True), t)
        t = np.concatenate([np.zeros((len(t), 1)), t], axis=1)
        mid = 0.5 * (t[:, 1:] + t[:, :-1])
        idx = [np.floor((r[:, a:a + 1] + mid * k[:, a:a + 1] + HALF) / (2 * HALF / n)).astype(np.int64) for a in range(3)]
        inside = np.all([(q >= 0) & (q < n) for q in idx], axis=0)
        q = [np.clip(v, 0, n - 1) for v in idx]
        tau[s:s + 4096] = SEXT * np.where(inside, dens[q[0], q[1], q[2]] * (t[:, 1:] - t[:, :-1]), 0.0).sum(axis=1)
    return tau


def _exact_tau_octree(case, seed):
    lev, pos, flags, dens = _tree(case, seed)
    lev, pos = lev[~flags], pos[~flags]
    top = int(lev.max())
    cell = np.zeros((1 << top,) * 3, np.int32)
    for level in range(top + 1):
        at = np.flatnonzero(lev == level)
        if len(at):
            n, s = 1 << level, 1 << (top - level)
            view = cell.reshape(n, s, n, s, n, s)
            view[pos[at, 0], :, pos[at, 1], :, pos[at, 2], :] = at[:, None, None, None]
    side = 2 * HALF / (1 << lev.astype(np.int64))
    lo = pos * side[:, None] - HALF
    rays = _rays(case, seed)
    r, k = rays[:, :3].copy(), rays[:, 3:]
    with np.errstate(divide="ignore", invalid="ignore"):
        near = np.where(np.abs(k) > 1e-15, (np.where(k > 0, -HALF, HALF) - r) / k, -np.inf)
        near[(np.abs(k) <= 1e-15) & (np.abs(r) > HALF)] = np.inf
    near = np.maximum(near.max(axis=1), 0.0)
    tau = np.zeros(len(r))
    live = np.flatnonzero(np.isfinite(near))
    p = r[live] + near[live, None] * k[live]
    eps, fine = 1e-11 * HALF, 2 * HALF / (1 << top)
    while len(live):
        d = k[live]
        ijk = np.floor((p + eps * d + HALF) / fine).astype(np.int64)
        ok = np.all((ijk >= 0) & (ijk < (1 << top)), axis=1)
        live, p, d, ijk = live[ok], p[ok], d[ok], ijk[ok]
        if not len(live):
            break
        c = cell[ijk[:, 0], ijk[:, 1], ijk[:, 2]]
        with np.errstate(divide="ignore", invalid="ignore"):
            t = np.where(np.abs(d) > 1e-15, (np.where(d > 0, lo[c] + side[c, None], lo[c]) - p) / d, np.inf).min(axis=1)
        t = np.maximum(t, 0.0)
        tau[live] += SEXT * dens[c] * t
        p = p + t[:, None] * d
    return tau


def _philox(c0, c1, c2, c3, k0, k1):
    """Philox4x32-10 (Salmon, Moraes, Dror & Shaw 2011) on uint64 arrays of 32-bit words."""
    low = np.uint64(0xFFFFFFFF)
    for r in range(10):
        a, b = np.uint64(0xD2511F53) * c0, np.uint64(0xCD9E8D57) * c2
        c0, c1, c2, c3 = ((b >> np.uint64(32)) ^ c1 ^ np.uint64(k0)) & low, b & low, ((a >> np.uint64(32)) ^ c3 ^ np.uint64(k1)) & low, a & low
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return c0, c1, c2, c3


def _exact_density(case, seed):
    n, samples = case["size"], case["samples"]
    b = _borders(n)
    m = np.arange(n ** 3)
    ijk = (m // (n * n), (m // n) % n, m % n)
    lo, hi = [b[q] for q in ijk], [b[q + 1] for q in ijk]
    phase = 2 * math.pi * np.random.default_rng(seed).random()
    key = seed + 3
    cell = m.astype(np.uint64)
    zero, draws, at = np.zeros_like(cell), [], []
    total = np.zeros(len(m))
    rho0 = 1.0 / (4 * math.pi * HR * HR * HZ)
    for block in range((3 * samples + 1) // 2):
        w = _philox(cell, zero, zero + np.uint64(block), zero + np.uint64(0x44454E53), key & 0xFFFFFFFF, key >> 32)
        for hi32, lo32 in ((w[0], w[1]), (w[2], w[3])):
            draws.append((((hi32 << np.uint64(20)) ^ (lo32 >> np.uint64(12))).astype(np.float64) + 0.5) * 2.0 ** -52)
        while len(draws) >= 3 and len(at) < samples:
            x, y, z = (lo[a] + draws[a] * (hi[a] - lo[a]) for a in range(3))
            draws = draws[3:]
            at.append(0)
            R = np.sqrt(x * x + y * y)
            v = rho0 * np.exp(-R / HR - np.abs(z) / HZ)
            if case["spiral"]:
                arm = np.log(R / (3 * PC)) / math.tan(math.radians(15.0)) + phase + 0.25 * math.pi - np.arctan2(y, x)
                v *= 0.5 + 0.5 * 2.0 * np.sin(arm) ** 2
            total += v
    return 5.0 / SEXT / (2 * rho0 * HZ) * total / samples


def _exact_guide(case, seed):
    """Loss and gradient of the von Mises-Fisher mixture network in 64 bits."""
    theta = torch.tensor(_theta(seed), dtype=torch.float64, requires_grad=True)
    rec = torch.tensor(_records(case, seed), dtype=torch.float64)
    h, at = rec[:, :9], 0
    for i, (nin, nout) in enumerate(((9, 64), (64, 64), (64, 64), (64, 40))):
        w, bias = theta[at:at + nin * nout].view(nout, nin), theta[at + nin * nout:at + nin * nout + nout]
        at += nin * nout + nout
        h = h @ w.T + bias
        if i < 3:
            h = torch.relu(h)
    o = h.view(-1, 8, 5)
    mu = o[..., :3] / o[..., :3].norm(dim=-1, keepdim=True).clamp_min(1e-12)
    kappa = torch.clamp(0.2 + torch.nn.functional.softplus(o[..., 3]), max=400.0)
    c = (mu * rec[:, None, 9:12]).sum(-1)
    f = kappa / (2 * math.pi * -torch.expm1(-2 * kappa)) * torch.exp(kappa * (c - 1))
    loss = -(rec[:, 12] * torch.log((torch.softmax(o[..., 4], dim=-1) * f).sum(-1))).sum()
    loss.backward()
    return {"grad": theta.grad.numpy(), "loss": loss.item()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "guide":
        return _exact_guide(case, seed)
    if kind == "tau" and case["grid"] in ("cartesian", "octree"):
        tau = _exact_tau_cartesian(case, seed) if case["grid"] == "cartesian" else _exact_tau_octree(case, seed)
        return {"path": tau, "obs": np.where(tau >= 745.0, np.inf, tau)}
    if kind == "density" and case["grid"] == "cartesian" and case["size"] ** 3 * case["samples"] <= 12_000_000:
        return _exact_density(case, seed)
    # the images of a Monte Carlo run have no value in closed form, and the segments and densities
    # on the meshes follow from the engine's own tables
    return None

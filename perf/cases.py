"""The work that users of this framework have it do, as cases that can be timed and compared.

A case is one whole simulation step through the public classes of skirt7_amd: photon-packet transport over
each kind of dust grid, in both precisions, read out as a user reads it (frames, absorption tables), a fitting
population in one batched run, a panchromatic run with dust emission, and optical depths along given rays.
The setups are those of skirt7_amd.workloads, with sizes from a first try-out to a production step.

listed() returns the cases, draw(rng) one more of the same ranges, prepare(case, seed) what a program holds
before the call (grid, media, instruments, simulation), run(state) one pass and its outputs, work(case) the
bytes and operations a pass cannot do without, exact(case, seed) the outputs in plain 64-bit numpy where they
have such a value (a Monte Carlo image has none: it is defined by the packets' random streams).
"""
import math

import numpy as np

from skirt7_amd import panchromatic
from skirt7_amd import skirt as S
from skirt7_amd import workloads
from skirt7_amd.capi import SG_FP64, SG_MIXED

PRECISION = {"fp64": SG_FP64, "mixed": SG_MIXED}


def listed():
    return [
        # a first try-out or a unit test of a ski file: few packets on a small grid, the default precision;
        # launches and latency are all there is
        {"name": "cart_small", "kind": "cartesian", "grid_n": 24, "pixels": 64, "packages": 5000, "tau": 1.0,
         "precision": "fp64"},
        # the plain oligochromatic galaxy at the reference's default of 1e6 packets, the default precision
        {"name": "cart_disc", "kind": "cartesian", "grid_n": 50, "pixels": 256, "packages": 1000000, "tau": 1.0,
         "precision": "fp64"},
        # the same galaxy as an interactive preview: mixed precision, ragged sizes, an optically thin disc
        {"name": "cart_preview", "kind": "cartesian", "grid_n": 63, "pixels": 201, "packages": 150001, "tau": 0.3,
         "precision": "mixed"},
        # a step of a production image: the spiral galaxy on its full octree (7e5 leaves, four 512^2 frames)
        {"name": "octree_large", "kind": "octree", "maxlevel": 8, "massfraction": 1e-6, "pixels": 512,
         "packages": 4000000, "tau": 2.0, "precision": "mixed"},
        # one model of a parameter study: a coarser octree, fewer packets
        {"name": "octree_mid", "kind": "octree", "maxlevel": 6, "massfraction": 1e-5, "pixels": 256,
         "packages": 200000, "tau": 0.5, "precision": "mixed"},
        # a reference run in the exact arithmetic, optically thick
        {"name": "octree_fp64", "kind": "octree", "maxlevel": 7, "massfraction": 1e-5, "pixels": 300,
         "packages": 300000, "tau": 5.0, "precision": "fp64"},
        # a Voronoi mesh with the absorption table over several wavelengths (input of dust heating)
        {"name": "voronoi_heating", "kind": "voronoi", "nsites": 100000, "nlambda": 3, "pixels": 256,
         "packages": 100000, "precision": "mixed"},
        # a hydrodynamic snapshot: a kd-tree over SPH particles, eight views
        {"name": "kdtree_particles", "kind": "kdtree", "particles": 500000, "massfraction": 1.8e-6, "pixels": 512,
         "packages": 500000, "precision": "mixed"},
        # one generation of a fit: uneven galaxies, each with its own grid and packet count, in one batched run
        {"name": "population", "kind": "population", "members": 24, "grid_n": 96, "min_packages": 1e5,
         "max_packages": 1e6, "precision": "mixed"},
        # two dust components with their own mixes, absorption stored, two wavelengths
        {"name": "two_dust", "kind": "two_dust", "grid": "octree", "size": 6, "pixels": 100, "packages": 100000,
         "precision": "mixed"},
        # a panchromatic galaxy: stellar emission at every wavelength, dust spectra, dust emission
        {"name": "panchromatic", "kind": "pan", "grid": "cartesian", "size": 24, "nlambda": 30, "pixels": 48,
         "packages": 20000, "precision": "mixed"},
        # an optical-depth map and the paths to given depths, along rays through a Cartesian grid
        {"name": "ray_map", "kind": "rays", "grid_n": 64, "rays": 200000, "tau": 2.0, "precision": "mixed"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cartesian", "cartesian", "octree", "octree", "voronoi", "kdtree", "population", "two_dust",
                       "pan", "rays"])
    precision = rng.choice(["fp64", "mixed", "mixed"])
    tau = round(math.exp(rng.uniform(math.log(0.1), math.log(5.0))), 3)
    if kind == "cartesian":
        return {"kind": kind, "grid_n": _log_int(rng, 8, 100), "pixels": rng.randint(24, 320),
                "packages": _log_int(rng, 2000, 1000000), "tau": tau, "precision": precision}
    if kind == "octree":
        return {"kind": kind, "maxlevel": rng.randint(4, 7), "massfraction": 10.0 ** rng.uniform(-5.5, -4.0),
                "pixels": rng.randint(32, 400), "packages": _log_int(rng, 5000, 300000 if precision == "fp64" else 2000000),
                "tau": tau, "precision": precision}
    if kind == "voronoi":
        return {"kind": kind, "nsites": _log_int(rng, 4000, 100000), "nlambda": rng.randint(1, 4),
                "pixels": rng.randint(32, 256), "packages": _log_int(rng, 5000, 75000), "precision": precision}
    if kind == "kdtree":
        return {"kind": kind, "particles": _log_int(rng, 40000, 400000), "massfraction": 10.0 ** rng.uniform(-5.6, -4.5),
                "pixels": rng.randint(64, 512), "packages": _log_int(rng, 5000, 100000 if precision == "fp64" else 400000),
                "precision": precision}
    if kind == "population":
        return {"kind": kind, "members": rng.randint(3, 24), "grid_n": rng.randint(33, 96), "min_packages": 2e4,
                "max_packages": 5e5, "precision": precision}
    if kind == "two_dust":
        grid = rng.choice(["cartesian", "octree", "voronoi"])
        size = {"cartesian": rng.randint(10, 48), "octree": rng.randint(4, 6), "voronoi": _log_int(rng, 2000, 30000)}[grid]
        return {"kind": kind, "grid": grid, "size": size, "pixels": rng.randint(24, 128),
                "packages": _log_int(rng, 5000, 80000), "precision": precision}
    if kind == "pan":
        grid = rng.choice(["cartesian", "octree"])
        return {"kind": kind, "grid": grid, "size": rng.randint(10, 30) if grid == "cartesian" else rng.randint(3, 5),
                "nlambda": rng.randint(12, 30), "pixels": rng.randint(16, 64), "packages": _log_int(rng, 2000, 20000),
                "precision": precision}
    return {"kind": "rays", "grid_n": _log_int(rng, 12, 100), "rays": _log_int(rng, 1000, 500000), "tau": tau,
            "precision": precision}


def _rays(case, seed):
    """Rays as an observer's raster sends them: origins on a plane outside the grid's box and inside it,
    directions spread over the sphere, and the optical depths to reach along each."""
    rng = np.random.default_rng(seed)
    n = case["rays"]
    k = rng.standard_normal((n, 3))
    k /= np.linalg.norm(k, axis=1)[:, None]
    r = rng.uniform(-1.0, 1.0, (n, 3)) * np.array([12.0, 12.0, 1.0])
    outside = rng.random(n) < 0.5
    r[outside] -= 60.0 * k[outside]
    return np.concatenate([r, k], axis=1), rng.exponential(0.3 * case["tau"], n)


def prepare(case, seed):
    kind = case["kind"]
    seed = 1 + seed % (2**31 - 1)
    n = case.get("packages")
    if kind == "cartesian":
        w = workloads.disc_cartesian(grid_n=case["grid_n"], pixels=case["pixels"], packages=n, seed=seed, nsamples=20,
                                     tau=case["tau"])
    elif kind == "octree":
        w = workloads.spiral_octree(tau=case["tau"], maxlevel=case["maxlevel"], pixels=case["pixels"], packages=n,
                                    seed=seed, maxmassfraction=case["massfraction"])
    elif kind == "voronoi":
        w = workloads.spiral_voronoi(nsites=case["nsites"], nlambda=case["nlambda"], pixels=case["pixels"], packages=n,
                                     seed=seed)
    elif kind == "kdtree":
        w = workloads.lognormal_kdtree(nvox=64, maxmassfraction=case["massfraction"], pixels=case["pixels"], packages=n,
                                       seed=seed, particles=case["particles"])
    elif kind == "population":
        p = workloads.fit_population(members=case["members"], packets=(case["min_packages"], case["max_packages"]),
                                     grid_n=(32, case["grid_n"]), seed=seed)
        return dict(kind=kind, precision=PRECISION[case["precision"]], members=p["members"],
                    counts=[int(m["packages"]) for m in p["members"]])
    elif kind == "two_dust":
        # the grid is frozen (its subdivision and sites come from the default seed), the packets are the seed's
        w = workloads.two_dust_disc(kind=case["grid"], grid_n=case["size"], maxlevel=case["size"], nsites=case["size"],
                                    pixels=case["pixels"], packages=n)
        w["sim"] = S.OligoMonteCarloSimulation(w["dust"], w["stars"], w["instr"], packages=n, seed=seed)
    elif kind == "pan":
        w = workloads.pan_disc(kind=case["grid"], nlambda=case["nlambda"], grid_n=case["size"], maxlevel=case["size"],
                               pixels=case["pixels"], packages=n)
        w["pan"] = panchromatic.PanMonteCarloSimulation(w["stars"], w["pan"].dust, w["instr"], packages=n, seed=seed,
                                                        precision=PRECISION[case["precision"]])
    else:
        w = workloads.disc_cartesian(grid_n=case["grid_n"], pixels=16, packages=1000, seed=4357, nsamples=8,
                                     tau=case["tau"])
        w["rk"], w["taus"] = _rays(case, seed)
    w["kind"] = kind
    w["precision"] = PRECISION[case["precision"]]
    return w


def _frames(instr):
    return [instr.frame(i) for i in range(len(instr.instruments))]


def run(state):
    kind = state["kind"]
    if kind == "population":
        for m in state["members"]:
            m["instr"].clear()
        S.run_batch([m["sim"] for m in state["members"]], state["counts"], precision=state["precision"])
        return [f for m in state["members"] for f in _frames(m["instr"])]
    if kind == "rays":
        dust = state["dust"]
        return [dust.opticaldepths(state["rk"], precision=state["precision"]),
                dust.pathlengths(state["rk"], state["taus"], precision=state["precision"])]
    if kind == "pan":
        pan = state["pan"]
        pan.runSelf()
        return _frames(state["instr"]) + [pan.Labs_stellar, pan.Labsbol]
    state["instr"].clear()
    stored = state["dust"].storeabsorptionrates()
    if stored:
        state["dust"].clear()
    state["sim"].runstellaremission(state["precision"])
    return _frames(state["instr"]) + ([state["dust"].Labs()] if stored else [])


def work(case):
    """Bytes: the medium read once, frames and tables written once. Operations: packets, walks per packet and cells
    per walk (estimates of these setups) times the operations of a crossing: three wall distances, the
    smallest, the position and the optical depth; a Voronoi crossing tests about 15 planes."""
    kind = case["kind"]
    real = 8 if case["precision"] == "fp64" else 4
    if kind == "rays":
        cells = case["grid_n"] ** 3
        return {"bytes": float(cells * real + case["rays"] * (2 * 48 + 8 + 16)),
                "flops": 2.0 * case["rays"] * case["grid_n"] * 30.0}
    views, nlambda, tau, per_crossing, tables = 3, 1, case.get("tau", 1.0), 30.0, 0
    packages, pixels = case.get("packages", 0), case.get("pixels", 0) ** 2
    if kind == "cartesian":
        cells, along, cell_bytes = case["grid_n"] ** 3, 0.8 * case["grid_n"], real
    elif kind == "octree":
        cells = min(8.0 ** case["maxlevel"], 0.8 / case["massfraction"])
        along, cell_bytes, views = 0.8 * cells ** (1.0 / 3.0), 8 * real, 4
    elif kind == "voronoi":
        cells, nlambda, views, tables = case["nsites"], case["nlambda"], 2, 1
        along, cell_bytes, per_crossing = 0.6 * cells ** (1.0 / 3.0), 450, 450.0
    elif kind == "kdtree":
        cells, views = 1.4 / case["massfraction"], 8
        along, cell_bytes = 0.8 * cells ** (1.0 / 3.0), 8 * real
    elif kind == "population":
        g = 0.5 * (32 + case["grid_n"])
        lo, hi = case["min_packages"], case["max_packages"]
        cells, along, cell_bytes, views = case["members"] * g ** 3, 0.8 * g, real, 1
        packages, pixels = case["members"] * (hi - lo) / math.log(hi / lo), case["members"] * 256 * 128
    else:
        cells = {"cartesian": case["size"] ** 3, "octree": min(8.0 ** case["size"], 8.0e3 * case["size"]),
                 "voronoi": case["size"]}[case["grid"]]
        along, cell_bytes, tables = 0.8 * cells ** (1.0 / 3.0), 2 * real, 1
        nlambda, views = (2, 3) if kind == "two_dust" else (2 * case["nlambda"], 2)
    scatterings = 0.5 + min(tau, 5.0)
    walks = packages * nlambda * ((views + 1) + scatterings * (views + 2))
    return {"bytes": float(cells * cell_bytes + (views * pixels + tables * cells) * nlambda * 8),
            "flops": float(walks * along * per_crossing)}


def _exact_rays(case, seed):
    """Optical depths and path lengths by sorting each ray's crossings with all cell borders: segment by segment
    density times length, and the linear inversion of the cumulative depth at the given one."""
    w = prepare(case, seed)
    borders = [np.asarray(v, np.float64) for v in (w["grid"].xv, w["grid"].yv, w["grid"].zv)]
    n = [len(v) - 1 for v in borders]
    rho = np.asarray(w["rho"], np.float64).reshape(n) * float(w["mix"].kappaext[0])
    taus_out, paths = [], []
    for lo in range(0, len(w["rk"]), 4096):
        r, k = w["rk"][lo:lo + 4096, :3], w["rk"][lo:lo + 4096, 3:]
        with np.errstate(divide="ignore"):
            s = [(borders[a][None, :] - r[:, a:a + 1]) / k[:, a:a + 1] for a in range(3)]
        enter = np.max([np.minimum(t[:, 0], t[:, -1]) for t in s], axis=0).clip(0.0)
        leave = np.min([np.maximum(t[:, 0], t[:, -1]) for t in s], axis=0)
        hit = leave > enter
        enter, leave = np.where(hit, enter, 0.0), np.where(hit, leave, 0.0)
        cuts = np.sort(np.clip(np.concatenate(s + [enter[:, None], leave[:, None]], axis=1), enter[:, None],
                               leave[:, None]), axis=1)
        mid, ds = 0.5 * (cuts[:, 1:] + cuts[:, :-1]), np.diff(cuts, axis=1)
        idx = [np.clip(np.searchsorted(borders[a], r[:, a:a + 1] + mid * k[:, a:a + 1], side="right") - 1, 0, n[a] - 1)
               for a in range(3)]
        tau = np.cumsum(np.where(hit[:, None], rho[idx[0], idx[1], idx[2]] * ds, 0.0), axis=1)
        target = w["taus"][lo:lo + 4096]
        j = np.minimum(np.sum(tau <= target[:, None], axis=1), tau.shape[1] - 1)
        rows = np.arange(len(j))
        t1 = tau[rows, j]
        t0 = np.where(j > 0, tau[rows, np.maximum(j - 1, 0)], 0.0)
        frac = np.where(t1 > t0, (target - t0) / np.where(t1 > t0, t1 - t0, 1.0), 0.0)
        taus_out.append(tau[:, -1])
        paths.append(np.where(~hit, 0.0, np.where(target > tau[:, -1], leave, cuts[rows, j] + frac * ds[rows, j])))
    return [np.concatenate(taus_out), np.concatenate(paths)]


def exact(case, seed):
    return _exact_rays(case, seed) if case["kind"] == "rays" else None

"""The work that users have this package do, as cases that can be timed.

Every case goes through a public entry point with host data in and host data
out, as a user's script calls it: ``mcxcl_amd.run`` (forward runs, records,
packed media, RF, adjoint outputs), ``mcxcl_amd.pmcxcl.Batch`` (many small
simulations in one launch), ``mcxcl_amd.autograd.detector_signals`` (a training
step's forward and backward) and ``signal_jacobians`` (an inversion's matrix).
The domains, media and photon counts follow ``mcxcl_amd.workloads`` and
``bench.py``; odd and ragged grids come with them.

A run with the default arithmetic (``mathmode`` 0) is a Monte Carlo estimate:
which lane runs which photon is settled while it runs, so two correct programs
agree only within the statistical error of their photon counts.  The photon
counts here are large enough for that error to stay below a percent or so of
the field's 2-norm.  The number of detected photons is itself random there, so
the records of such a run have no fixed shape; they come back whole in the
cases with bit-reproducible arithmetic (``mathmode`` 1), where the photons are
the same in every run and only the order of the records is free.
"""

import math

import numpy as np
import torch

import mcxcl_amd
from mcxcl_amd import autograd, pmcxcl, workloads

# operations of one photon event in the transport algebra (bench.py's model)
OPS_STEP, OPS_DEPOSIT, OPS_SCATTER = 65.0, 17.0, 135.0

SOFT = {"cube": (0.005, 1.0), "sphere": (0.005, 1.2), "layers": (0.015, 8.0)}   # typical mua, mus (1/mm)


def listed():
    return [
        # the smallest call: a few photons with their records and seeds, bit-reproducible
        # (a regression check, the set-up of a replay), where staging and launches count
        {"name": "records_sphere60_2e4", "kind": "records", "volume": "sphere", "nx": 60, "ny": 60, "nz": 60,
         "source": "pencil", "photons": 20000, "gates": 10, "detectors": 4, "reflect": 1},
        # a quick look at a new set-up, the inner call of a fit: a pencil beam into the 60^3 cube
        {"name": "cube60_pencil_3e5", "kind": "forward", "volume": "cube", "nx": 60, "ny": 60, "nz": 60,
         "source": "pencil", "photons": 300000, "gates": 1, "detectors": 0, "reflect": 1},
        # an everyday run: the sphere-in-cube, ten time gates, detectors on
        {"name": "sphere60_pencil_1e6", "kind": "forward", "volume": "sphere", "nx": 60, "ny": 60, "nz": 60,
         "source": "pencil", "photons": 1000000, "gates": 10, "detectors": 4, "reflect": 1},
        # the benchmark workload at its full photon count
        {"name": "sphere60_pencil_1e8", "kind": "forward", "volume": "sphere", "nx": 60, "ny": 60, "nz": 60,
         "source": "pencil", "photons": 100000000, "gates": 10, "detectors": 4, "reflect": 1},
        # wide-field illumination (cube60planar): the general launch, deposits spread over the grid
        {"name": "cube60_planar_1e7", "kind": "forward", "volume": "cube", "nx": 60, "ny": 60, "nz": 60,
         "source": "planar", "photons": 10000000, "gates": 1, "detectors": 0, "reflect": 1},
        # a segmented volume whose voxels carry their own mua and mus as two halves,
        # an isotropic point inside it (an implanted fibre), a ragged grid
        {"name": "halves_isotropic_71x64x53", "kind": "halves", "volume": "sphere", "nx": 71, "ny": 64, "nz": 53,
         "source": "isotropic", "photons": 3000000, "gates": 1, "detectors": 0, "reflect": 1},
        # a head-like layered volume at 1 mm, forward fluence and detection
        {"name": "layers200_pencil_1e7", "kind": "forward", "volume": "layers", "nx": 200, "ny": 200, "nz": 200,
         "source": "pencil", "photons": 10000000, "gates": 1, "detectors": 8, "reflect": 1},
        # a step of an absorption fit: detector signals of per-voxel media and their gradient
        {"name": "gradient_layers100_1e7", "kind": "gradient", "volume": "layers", "nx": 100, "ny": 100, "nz": 100,
         "photons": 10000000, "gates": 1, "detectors": 8, "reflect": 1},
        # the sensitivity matrix of a source-detector array, mua and mus, reproducible photons
        {"name": "jacobians_48_4x4", "kind": "jacobians", "nx": 48, "ny": 48, "nz": 48, "side": 2,
         "photons": 2000000},
        # a parameter study: independent small domains in one launch, one step of a kept batch
        {"name": "batch_16x48", "kind": "batch", "instances": 16, "dim": 48, "photons": 400000},
        # frequency-domain light (150 MHz): complex fluence
        {"name": "rf_sphere60_3e6", "kind": "rf", "volume": "sphere", "nx": 60, "ny": 60, "nz": 60,
         "source": "pencil", "photons": 3000000, "gates": 10, "detectors": 4, "reflect": 1},
        # adjoint Jacobians (mua and D) from the fluences of sources and detectors
        {"name": "adjoint_96_2x2", "kind": "adjoint", "nx": 96, "ny": 96, "nz": 96, "side": 2, "photons": 1000000},
    ]


def _between(rng, low, high):
    """a whole number, its logarithm uniform"""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["forward", "forward", "forward", "halves", "gradient", "jacobians", "batch", "rf", "adjoint",
                       "records"])
    case = {"kind": kind}

    if kind == "batch":
        case.update(instances=_between(rng, 4, 16), dim=_between(rng, 24, 56), photons=_between(rng, 300000, 500000))
        return case

    if kind in ("jacobians", "adjoint"):
        case.update({d: _between(rng, 24, 80) for d in ("nx", "ny", "nz")})
        case.update(side=rng.choice([1, 2]), photons=_between(rng, 100000, 2000000))
        return case

    case["volume"] = "layers" if kind == "gradient" else rng.choice(["cube", "sphere", "layers"])
    high = 160 if case["volume"] == "layers" else 100
    case.update({d: _between(rng, 30, high) for d in ("nx", "ny", "nz")})
    case["gates"] = 1 if kind in ("gradient", "halves") else _between(rng, 1, 12)
    case["reflect"] = 1 if kind == "gradient" else rng.choice([1, 1, 0])

    if kind == "gradient":
        case.update(photons=_between(rng, 3000000, 10000000), detectors=8)
        return case

    case["source"] = rng.choice(["pencil", "isotropic", "disk"] + (["planar"] if kind == "forward" else []))
    case["detectors"] = rng.choice([0, 4]) if kind != "records" else 4

    if kind == "records":
        case["photons"] = _between(rng, 20000, 3000000)
    elif case["source"] == "planar":
        case.update({d: min(case[d], 80) for d in ("nx", "ny", "nz")}, photons=_between(rng, 10000000, 20000000))
    else:
        low = {"pencil": 300000, "isotropic": 1000000, "disk": 2000000}[case["source"]]
        case["photons"] = _between(rng, low, 10000000 if kind == "forward" else 3000000)

    return case


def _labels(case, rng):
    """label volume and property table of a case's geometry"""
    shape = (case["nx"], case["ny"], case["nz"])

    if case["volume"] == "layers":
        dim = max(shape)
        depths = [max(1, int(case["nz"] * f)) for f in (0.1, 0.2, 0.35)]
        vol = workloads.layered_volume(dim, depths, 0.04 * case["nz"], int(rng.integers(1 << 30)))
        vol = np.asfortranarray(vol[:shape[0], :shape[1], :shape[2]])
        prop = np.array(workloads.LAYER_PROP, np.float32)
    else:
        vol = np.ones(shape, np.uint8, order="F")
        prop = np.array(workloads.CUBE60_PROP, np.float32)

        if case["volume"] == "sphere":
            centre = [0.5 * n + rng.uniform(-2, 2) for n in shape]
            radius = 0.25 * min(shape)
            d2 = sum(np.square(np.arange(n) + 0.5 - c).reshape([-1 if i == k else 1 for k in range(3)])
                     for i, (n, c) in enumerate(zip(shape, centre)))
            vol[d2 <= radius * radius] = 2

    prop[1:, :2] *= rng.uniform(0.97, 1.03, prop[1:, :2].shape).astype(np.float32)
    return vol, prop


def _config(case, rng):
    """the run's dict for mcxcl_amd.run"""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    vol, prop = _labels(case, rng)
    cx, cy = float(nx // 2), float(ny // 2)
    cfg = {"nphoton": case["photons"], "vol": vol, "prop": prop, "tstart": 0.0, "tend": 5e-9,
           "tstep": 5e-9 / case["gates"], "srcpos": [cx, cy, 0.0], "srcdir": [0, 0, 1],
           "isreflect": case["reflect"], "issrcfrom0": 1, "seed": int(rng.integers(1, 1 << 30)), "issavedet": 0}
    source = case.get("source", "pencil")

    if source == "isotropic":
        cfg.update(srctype="isotropic", srcpos=[cx + 0.3, cy - 0.2, nz / 3.0 + 0.4])
    elif source == "disk":
        cfg.update(srctype="disk", srcparam1=[min(nx, ny) / 12.0, 0, 0, 0])
    elif source == "planar":
        # the middle two thirds of the face, from 10 voxels above it (cube60planar)
        cfg.update(srctype="planar", srcpos=[nx / 6.0, ny / 6.0, -10.0], srcparam1=[nx * 2 / 3.0, 0, 0, 0],
                   srcparam2=[0, ny * 2 / 3.0, 0, 0])

    if case["detectors"]:
        ring = [2 * math.pi * i / case["detectors"] for i in range(case["detectors"])]
        away = max(4.0, min(nx, ny) / (10.0 if case["kind"] == "gradient" else 6.0))
        cfg.update(issavedet=1, savedetflag="DPX", maxdetphoton=4000000,
                   detpos=[[cx + away * math.cos(a), cy + away * math.sin(a), 0, 2.0] for a in ring])

    return cfg


def _array(case, rng):
    """a side x side array of pencil sources with as many detectors between them on the top face"""
    nx, ny, nz, side = case["nx"], case["ny"], case["nz"], case["side"]
    sx, sy = nx / (side + 0.5), ny / (side + 0.5)
    at = [(i, j) for j in range(side) for i in range(side)]
    vol = np.ones((nx, ny, nz), np.uint8, order="F")
    vol[:, :, nz // 4:] = 2
    prop = np.array([[0, 0, 1, 1], [0.01, 2.0, 0.8, 1.37], [0.02, 3.0, 0.8, 1.37]], np.float32)
    prop[1:, :2] *= rng.uniform(0.9, 1.1, (2, 2)).astype(np.float32)
    return {"nphoton": case["photons"], "vol": vol, "prop": prop, "tstart": 0.0, "tend": 5e-9, "tstep": 5e-9,
            "srcpos": [[sx * (i + 0.5), sy * (j + 0.5), 0] for i, j in at], "srcdir": [[0, 0, 1, 0]] * len(at),
            "detpos": [[sx * (i + 1.0), sy * (j + 1.0), 0, 2] for i, j in at], "isreflect": 1, "issrcfrom0": 1,
            "seed": int(rng.integers(1, 1 << 30)), "mathmode": 1}


def prepare(case, seed):
    rng = np.random.default_rng(int(seed))
    kind = case["kind"]

    if kind == "batch":
        n = case["photons"]
        cfgs = workloads.batched_workload(case["instances"], case["dim"], int(rng.integers(1, 1 << 20)),
                                          (n, 4 * n))

        for cfg in cfgs:
            if cfg["srctype"] == "disk":
                cfg["srcparam1"] = [case["dim"] / 24.0, 0, 0, 0]

        return {"kind": kind, "batch": pmcxcl.Batch(cfgs)}

    if kind == "adjoint":
        cfg = _array(case, rng)
        cfg.update(outputtype="adjoint_mua_d", detdir=[[0, 0, 1, 0]] * len(cfg["detpos"]), issavedet=0)
        return {"kind": kind, "cfg": cfg}

    if kind == "jacobians":
        cfg = _array(case, rng)

        if case["side"] == 1:
            cfg.update(srcpos=cfg["srcpos"][0], srcdir=cfg["srcdir"][0])

        cfg.update(savedetflag="DP", maxdetphoton=4000000)
        vol, prop = cfg["vol"], cfg["prop"]
        mua = prop[vol, 0] * (1 + 0.3 * rng.random(vol.shape, np.float32))
        mus = prop[vol, 1] * (1 + 0.3 * rng.random(vol.shape, np.float32))
        return {"kind": kind, "cfg": cfg, "mua": mua, "mus": mus}

    cfg = _config(case, rng)

    if kind == "rf":
        cfg.update(omega=2 * math.pi * 150e6)
    elif kind == "records":
        cfg.update(mathmode=1, issaveseed=1)
    elif kind == "halves":
        vol, prop = cfg["vol"], cfg["prop"]
        packed = np.empty((2,) + vol.shape, np.float32, order="F")
        packed[0], packed[1] = prop[vol, 0], prop[vol, 1]
        packed *= rng.uniform(0.9, 1.1, packed.shape).astype(np.float32)
        cfg.update(vol=packed, issavedet=0)
    elif kind == "gradient":
        cfg.update(savedetflag="DP")
        vol, prop = cfg["vol"], cfg["prop"]
        where = "cuda" if torch.cuda.is_available() else "cpu"
        mua = torch.tensor(np.ascontiguousarray(prop[vol, 0]), device=where, requires_grad=True)
        mus = torch.tensor(np.ascontiguousarray(prop[vol, 1]), device=where)
        weight = torch.tensor(rng.uniform(0.5, 1.5, case["detectors"]), device=where)
        return {"kind": kind, "cfg": cfg, "mua": mua, "mus": mus, "weight": weight}

    return {"kind": kind, "cfg": cfg}


def run(state):
    kind = state["kind"]

    if kind == "batch":
        state["batch"].run(1)
        return [{"flux": out["flux"], "launched": out["stat"]["energytot"]} for out in state["batch"].collect()]

    if kind == "gradient":
        mua = state["mua"]
        mua.grad = None
        signals = autograd.detector_signals(mua, state["mus"], state["cfg"])
        (signals * state["weight"]).sum().backward()
        return {"signals": signals.detach(), "gradient": mua.grad}

    if kind == "jacobians":
        signals, dmua, dmus = autograd.signal_jacobians(state["mua"], state["mus"], state["cfg"])
        return {"signals": signals, "dmua": dmua, "dmus": dmus}

    out = mcxcl_amd.run(state["cfg"])
    got = {"flux": out["flux"], "launched": out["stat"]["energytot"], "absorbed": out["stat"]["energyabs"]}

    if kind == "adjoint":
        got.update(jmua=out["jmua"], jd=out["jd"])
    elif kind == "records":
        # the records' order is free: sorted by detector, then by path and exit position,
        # in arrays of a fixed capacity (their number differs from seed to seed)
        cap = state["cfg"]["nphoton"] // 4
        detp, seeds = np.zeros((6, cap), np.float32), np.zeros((16, cap), np.uint8)

        if "detp" in out:
            order = np.lexsort(out["detp"][::-1])[:cap]
            detp[:, :order.size] = out["detp"][:, order]
            seeds[:, :order.size] = out["seeds"][:, order]

        got.update(detp=detp, seeds=seeds)

    return got


def work(case):
    """Operations: the mean path of a photon in a box is a few times its edge
    (4 volume/surface for diffuse light, longer with internal reflection and
    normal incidence: 130 mm measured in the 60^3 sphere-in-cube), capped by
    the 5 ns window; 1.5 voxel faces and mus scatterings per mm of it.  Bytes:
    one word per voxel in, the float32 outputs out."""
    kind = case["kind"]

    if kind == "batch":
        edge, mus, nvox = case["dim"], 10.0, case["instances"] * case["dim"] ** 3
        photons = case["instances"] * case["photons"] * 3 / math.log(4.0)
        out = nvox
    else:
        nvox = case["nx"] * case["ny"] * case["nz"]
        edge, photons = nvox ** (1.0 / 3.0), case["photons"]
        mus = SOFT[case["volume"]][1] if "volume" in case else 2.5
        pairs = case.get("side", 1) ** 4
        out = {"rf": 2 * case.get("gates", 1), "gradient": 1, "jacobians": 2 * pairs,
               "adjoint": 2 * pairs + 2 * case.get("side", 1) ** 2}.get(kind, case.get("gates", 1)) * nvox

    path = min(2.2 * edge, 1000.0)
    ops = 1.5 * (OPS_STEP + OPS_DEPOSIT) + mus * (OPS_STEP + OPS_SCATTER)
    return {"bytes": 4.0 * (nvox + out), "flops": photons * path * ops}


def tolerance(case):
    if case["kind"] in ("records", "adjoint", "jacobians"):
        # the same photons in every run: float64 sums in another order, rounded to float32
        return {"rel": 1e-5, "max": 1e-3}

    # four times the difference of two independent sets of photons: measured 7e-3 at
    # 1e6 photons of a pencil beam (6.8 / sqrt(photons); 5 to 8 over the volumes) and
    # up to 12 / sqrt(photons) from a point inside; 0.4 to 2 percent for the wider
    # sources, the batch and the gradient
    spread = {"pencil": 8.0, "isotropic": 12.0}.get(case.get("source"), 1e9)
    rel = min(0.03, 4.0 * spread / math.sqrt(case["photons"]))
    return {"rel": rel, "max": min(0.99, 60.0 * rel)}


def exact(case, seed):
    """What of a Monte Carlo run has a value in closed form: every photon is
    launched with unit weight."""
    if case["kind"] in ("gradient", "jacobians", "batch"):
        return None

    got = {"flux": None, "launched": float(case["photons"]), "absorbed": None}

    if case["kind"] == "adjoint":
        got.update(jmua=None, jd=None)
    elif case["kind"] == "records":
        got.update(detp=None, seeds=None)

    return got

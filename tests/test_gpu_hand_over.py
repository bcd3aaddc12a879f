"""Lanes that move between the waves of a workgroup, and fixed maps spread over
one-wave workgroups: photon counts at the edges of waves, workgroups and the
spread, and every kind of state that a lane takes along (launches, media,
records, replays), against the oracle on the same seeds and thread map.

A lane moves with its stream, tallies and index, so records and energies are
bit-exact; the float64 grid differs in the order of its sums only: fewer than
1e6 terms of one sign per voxel, each sum within 1e6 * 2^-53 < 1e-9 relative."""

import numpy as np
import pytest

import mcxcl_amd
import oracle
from helpers import sorted_records, sorted_seeds, split_sphere_volume
from mcxcl_amd import pmcxcl, workloads

pytestmark = pytest.mark.gpu

_DET = dict(issavedet=1, issaveseed=1, savedetflag="DSPMXVW")


@pytest.mark.parametrize("nphoton,nthread", [
    (1, 64), (63, 128), (65, 128), (257, 512), (1025, 1024), (16384, 16448),   # one-wave workgroups
    (16385, 16448), (66000, 66112), (70001, 66048),                            # 256-lane workgroups, ragged ends
])
def test_fixed_map_matches_oracle(nphoton, nthread):
    cfg = workloads.sphere_cube_workload(nphoton=nphoton, tend=1e-9, **_DET)
    cfg = dict(cfg, autopilot=0, nthread=nthread, nblocksize=64, mathmode=1, rawfield=1)
    gpu, ref = mcxcl_amd.run(cfg), oracle.run(cfg, nthread=nthread)
    assert gpu["stat"]["energytot"] == ref["stat"]["energytot"]
    assert gpu["stat"]["energyabs"] == ref["stat"]["energyabs"]
    np.testing.assert_allclose(gpu["flux64"], ref["flux64"], rtol=1e-9, atol=1e-12)
    assert ("detp" in gpu) == ("detp" in ref) and (nphoton < 1000 or "detp" in ref)
    if "detp" in ref:
        assert gpu["detp"].shape == ref["detp"].shape
        assert np.array_equal(sorted_records(gpu["detp"]), sorted_records(ref["detp"]))
        assert np.array_equal(sorted_seeds(gpu["seeds"]), sorted_seeds(ref["seeds"]))


NT = 2048
_LABELS = np.asarray([[0, 0, 1, 1], [0.005, 1.0, 0.01, 1.37], [0.02, 4.0, 0.5, 1.37]], np.float32)
_PATTERNS = np.random.default_rng(2024).uniform(0.2, 1.0, (2, 4, 3)).astype(np.float32)
_AREA = dict(srcpos=[10, 15, 0], srcparam1=[40, 0, 0, 4], srcparam2=[0, 30, 0, 3])
_OMEGA = 2 * np.pi * 150e6


def _sphere(nphoton=20000, **over):
    return workloads.sphere_cube_workload(nphoton=nphoton, **dict(dict(_DET, tstep=1e-9), **over))


def _pervoxel():
    vol = workloads.sphere_volume()
    pert = np.random.default_rng(7).uniform(0.7, 1.3, vol.shape).astype(np.float32)
    return np.stack([_LABELS[vol, 0] * pert, _LABELS[vol, 1] * (2 - pert)]).astype(np.float32)


def _labelplus():
    vol = workloads.sphere_volume()
    comp = np.random.default_rng(8).integers(0, 2, vol.shape)
    value = np.where(comp == 0, _LABELS[vol, 0], _LABELS[vol, 1])
    return np.stack([value, comp, vol]).astype(np.float32)


def _under_air():
    vol = workloads.sphere_volume().copy()
    vol[:, :, 0] = 0
    return vol


_BALL = dict(nphoton=20000, tstart=0, tend=5e-9, tstep=1e-9, srcpos=[20.5, 20.5, 0], srcdir=[0, 0, 1], issrcfrom0=1,
             isreflect=1, seed=99, issavedet=1, issaveseed=1, savedetflag="DSPMXV",
             detpos=[[26.5, 20.5, 7.35, 3.0], [14.5, 20.5, 7.35, 3.0]])
_POL = dict(nphoton=20000, vol=np.ones((30, 30, 20), np.uint8), prop=[[0, 0, 1, 1], [0.005, 0, 0, 1.33]],
            polprop=[[0.005, 0.3, 0.002, 1.59, 1.33]], srcpos=[15, 15, 0], srcdir=[0, 0, 1], srciquv=[1, 1, 0, 0],
            tstart=0, tend=5e-9, tstep=1e-9, seed=11, detpos=[[15, 15, 0, 6]], issavedet=1, isreflect=1, issaveseed=1)
_POL["lambda"] = 632.8

# what a lane carries besides the pencil path's state: the general launch's scratch, per-voxel
# properties, the complex weight, split planes, Stokes vectors, the pixel and weights of shared
# patterns, the source id, trajectory indices, the 2D and sampled-phase branches
STATES = {
    "planar": lambda: _sphere(srctype="planar", **_AREA),
    "planar without reflection": lambda: _sphere(srctype="planar", isreflect=0, **_AREA),
    "pervoxel": lambda: _sphere(muamus=_pervoxel(), savedetweight=1),
    "halves": lambda: _sphere(vol=_pervoxel(), prop=_LABELS.tolist()),
    "labelplus": lambda: _sphere(vol=_labelplus(), prop=_LABELS.tolist(), savedetflag="DXVW"),
    "rf": lambda: _sphere(omega=_OMEGA, minenergy=0.01),
    "svmc air": lambda: dict(_BALL, vol=split_sphere_volume(40, (20, 20, 20), 14, 1, 0),
                             prop=[[0, 0, 1, 1], [0.01, 1.0, 0.5, 1.37]]),
    "svmc tissue": lambda: dict(_BALL, vol=split_sphere_volume(40, (20, 20, 20), 12, 2, 1),
                                prop=[[0, 0, 1, 1], [0.01, 1.0, 0.5, 1.37], [0.03, 3.0, 0.8, 1.6]], issavedet=0),
    "polarised": lambda: dict(_POL),
    "polarised trajectories": lambda: dict(_POL, nphoton=2000, debuglevel="M", istrajstokes=1),
    "trajectories": lambda: _sphere(nphoton=3000, debuglevel="M"),
    "shared patterns": lambda: _sphere(srctype="pattern", srcnum=2, srcpattern=_PATTERNS, **_AREA),
    "shared patterns rf": lambda: _sphere(srctype="pattern", srcnum=2, srcpattern=_PATTERNS, omega=_OMEGA, **_AREA),
    "angles": lambda: _sphere(srcpos=[29.5, 29.5, 0], angleinvcdf=np.linspace(0, 0.45, 9).astype(np.float32)),
    "hyperboloid": lambda: _sphere(srctype="hyperboloid", srcpos=[30, 30, 0], srcparam1=[3, 10, 20, 0]),
    "sources pooled": lambda: _sphere(srcid=0, srcpos=[[29, 29, 0, 1], [12, 29, 0, 1]], srcdir=[[0, 0, 1, 0]] * 2),
    "sources apart": lambda: _sphere(srcid=-1, srcpos=[[29, 29, 0, 1], [12, 29, 0, 1]], srcdir=[[0, 0, 1, 0]] * 2),
    "reflectance": lambda: _sphere(vol=_under_air(), issaveref=1, issavedet=0),
    "flat": lambda: dict(_sphere(vol=np.ones((60, 60, 1), np.uint8), srcpos=[29.5, 0, 0.5], srcdir=[0, 1, 0]),
                         issavedet=0),
    "roulette and gscatter": lambda: _sphere(srctype="isotropic", srcpos=[29.5, 29.5, 29.5], minenergy=0.05, gscatter=3),
}


def _agree(gpu, ref, keys):
    for k in ("energytot", "energyabs"):
        assert gpu["stat"][k] == ref["stat"][k]
    scale = np.abs(ref["flux64"]).max()
    assert scale > 0
    np.testing.assert_allclose(gpu["flux64"], ref["flux64"], rtol=1e-9, atol=1e-12 * max(1.0, scale))
    for k in ("detp", "traj"):
        assert (k in gpu) == (k in ref) == (k in keys)
        if k in ref:
            assert gpu[k].shape == ref[k].shape and np.array_equal(sorted_records(gpu[k]), sorted_records(ref[k]))


def _keys(cfg):
    return [k for k, on in (("detp", cfg.get("issavedet")), ("traj", "debuglevel" in cfg)) if on]


@pytest.mark.parametrize("name", STATES)
def test_lane_state_moves_whole(name, monkeypatch):
    """the 256-lane workgroups of a large fixed map, every lane with ten photons (the moved
    lanes launch more of them) on this few lanes"""
    monkeypatch.setenv("MCXHIP_BLOCK", "256")
    cfg = dict(STATES[name](), autopilot=0, nthread=NT, nblocksize=64, mathmode=1, rawfield=1)
    ref = oracle.run(cfg, nthread=NT)
    _agree(mcxcl_amd.run(cfg), ref, _keys(cfg))


@pytest.mark.parametrize("name", ["planar", "rf", "svmc air", "polarised", "sources pooled"])
def test_lane_state_moves_whole_on_a_large_map(name):
    """the same workgroups as the launch plan chooses them: more lanes than the spread takes"""
    cfg = dict(STATES[name](), autopilot=0, nthread=20032, nblocksize=64, mathmode=1, rawfield=1)
    ref = oracle.run(cfg, nthread=20032)
    _agree(mcxcl_amd.run(cfg), ref, _keys(cfg))


@pytest.fixture(scope="module")
def recorded():
    cfg = _sphere(nphoton=100000, muamus=_pervoxel(), savedetweight=1, savedetflag="DSPM", ismomentum=1)
    return cfg, oracle.run(dict(cfg, autopilot=0, nthread=NT, nblocksize=64), nthread=NT)


@pytest.mark.parametrize("outputtype", ["jacobian", "wp", "wm", "rf", "rfmus", "wltof", "wptof"])
@pytest.mark.parametrize("replaydet", [0, -1])
def test_replays_move_whole(recorded, outputtype, replaydet, monkeypatch):
    monkeypatch.setenv("MCXHIP_BLOCK", "256")
    base, fwd = recorded
    assert fwd["detp"].shape[1] > 300
    cfg = dict(base, seed=fwd["seeds"], detphotons=fwd["detp"], replayweight=fwd["detw"], outputtype=outputtype,
               replaydet=replaydet, omega=_OMEGA, savedetweight=0, autopilot=0, nthread=NT, nblocksize=64, mathmode=1,
               rawfield=1)
    ref = oracle.run(cfg, nthread=NT)
    _agree(mcxcl_amd.run(cfg), ref, _keys(cfg))


@pytest.mark.parametrize("outputtype", ["jacobian", "wp", "wm", "rf", "rfmus", "wltof", "wptof"])
def test_fast_replays_move_whole(recorded, outputtype, monkeypatch):
    """the default arithmetic's replay on a fixed map, in 256-lane workgroups and in the spread
    that moves nothing: the same photons, so the grids differ by the float32 box's rounding
    alone (below 1e-6 of the whole)"""
    base, _ = recorded
    fwd = mcxcl_amd.run(dict(base, mathmode=0))
    assert fwd["detp"].shape[1] > 300
    cfg = dict(base, seed=fwd["seeds"], detphotons=fwd["detp"], replayweight=fwd["detw"], outputtype=outputtype,
               replaydet=0, omega=_OMEGA, savedetweight=0, mathmode=0, rawfield=1, rawonly=1)
    spread = mcxcl_amd.run(cfg)["flux64"]
    monkeypatch.setenv("MCXHIP_BLOCK", "256")
    moved = mcxcl_amd.run(cfg)["flux64"]
    size, err = np.linalg.norm(spread), np.linalg.norm(moved - spread)
    assert size > 0 and err <= 1e-6 * size


def _absorbed(out, n):
    """absorbed and deposited weight per photon"""
    return np.array([out["stat"]["energyabs"], out["flux64"].sum()]) / n


@pytest.mark.parametrize("nphoton", [1, 64, 1025, 262145])
@pytest.mark.parametrize("det", [False, True])
def test_run_time_hand_out_launches_every_photon(nphoton, det):
    """1024- and 768-lane workgroups; the launched weight is a sum of ones, exact in float32.
    Absorbed and deposited weight against a bit-reproducible run: a photon's share p lies in
    [0, 1], so its variance is at most p (1 - p)"""
    cfg = workloads.sphere_cube_workload(nphoton=nphoton, mathmode=0, outputtype="energy", rawfield=1,
                                         **(_DET if det else {}))
    out = mcxcl_amd.run(cfg)
    assert out["stat"]["energytot"] == nphoton
    p = _absorbed(mcxcl_amd.run(dict(cfg, nphoton=400000, mathmode=1)), 400000)
    assert (np.abs(_absorbed(out, nphoton) - p) <= 6 * np.sqrt(p * (1 - p) * (1 / nphoton + 1 / 400000))).all()


@pytest.mark.parametrize("blocksize", [64, 128, 320, 448, 1024])
def test_batch_workgroups_launch_every_photon(blocksize):
    """one to sixteen waves, with counts that do not divide by four; absorbed and deposited
    weight as above"""
    cfgs = [dict(c, outputtype="energy", rawfield=1)
            for c in workloads.batched_workload(ninst=3, dim=32, seed=5, photons=(1e4, 3e4))]
    for out, cfg in zip(pmcxcl.run_batch(cfgs, blocksize=blocksize)[0], cfgs):
        n = cfg["nphoton"]
        assert out["stat"]["energytot"] == n
        p = _absorbed(mcxcl_amd.run(dict(cfg, nphoton=200000, mathmode=1)), 200000)
        assert (np.abs(_absorbed(out, n) - p) <= 6 * np.sqrt(p * (1 - p) * (1 / n + 1 / 200000))).all()


def test_a_map_of_many_lanes_matches_oracle():
    """four times the default map's lanes; a short window keeps the oracle quick"""
    n = 2700000
    cfg = workloads.sphere_cube_workload(nphoton=n, tend=1e-10, tstep=1e-10, **_DET)
    cfg = dict(cfg, autopilot=0, nthread=n + 32, nblocksize=64, mathmode=1, rawfield=1)
    _agree(mcxcl_amd.run(cfg), oracle.run(cfg, nthread=n + 32), ["detp"])

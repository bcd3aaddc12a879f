"""Lanes that move between the waves of a workgroup, and fixed maps spread over
one-wave workgroups: photon counts at the edges of waves, workgroups and the
spread, against the oracle on the same seeds and thread map.

A lane moves with its stream, tallies and index, so records and energies are
bit-exact; the float64 grid differs in the order of its sums only: fewer than
1e6 terms of one sign per voxel, each sum within 1e6 * 2^-53 < 1e-9 relative."""

import numpy as np
import pytest

import mcxcl_amd
import oracle
from helpers import sorted_records, sorted_seeds
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


@pytest.mark.parametrize("nphoton", [1, 64, 1025, 262145])
@pytest.mark.parametrize("det", [False, True])
def test_run_time_hand_out_launches_every_photon(nphoton, det):
    """1024- and 768-lane workgroups; the launched weight is a sum of ones, exact in float32"""
    cfg = workloads.sphere_cube_workload(nphoton=nphoton, mathmode=0, **(_DET if det else {}))
    out = mcxcl_amd.run(cfg)
    assert out["stat"]["energytot"] == nphoton
    assert 0 <= out["stat"]["energyabs"] <= nphoton


@pytest.mark.parametrize("blocksize", [64, 128, 320, 448, 1024])
def test_batch_workgroups_launch_every_photon(blocksize):
    """one to sixteen waves, with counts that do not divide by four"""
    cfgs = workloads.batched_workload(ninst=3, dim=32, seed=5, photons=(1e4, 3e4))
    for out, cfg in zip(pmcxcl.run_batch(cfgs, blocksize=blocksize)[0], cfgs):
        assert out["stat"]["energytot"] == cfg["nphoton"]
        assert 0 < out["stat"]["energyabs"] < cfg["nphoton"]

"""Rounding of the default arithmetic's float32 deposit box.  A replay traces the same
photons on a fixed map, so a run without a box (MCXHIP_BOX_BYTES=0: every deposit is summed
in float64) gives the same deposits' sums, exact but for 1e-12.

A cell that is held within a limit R (a beam 256, a plane and a slit 32) errs by at most
2^-24 R an add, uniformly: N adds of mean w, together S = N w, differ from their sum by
2^-24 R / sqrt(3 S w) of it (one standard deviation; w is about 1/2 for path lengths in a
voxel).  Three of them are allowed, for what the lanes that deposit at the same time take a
cell past R.  A deposit far above R leaves at most R behind: 2^-24 of itself."""

import numpy as np
import pytest

import mcxcl_amd

pytestmark = pytest.mark.gpu

BEAM = dict(srcpos=[20, 20, 0], srcdir=[0, 0, 1])
PLANE = dict(srctype="planar", srcpos=[4, 4, 0], srcdir=[0, 0, 1], srcparam1=[32, 0, 0, 0], srcparam2=[0, 32, 0, 0])
SLIT = dict(PLANE, srcpos=[4, 20, 0], srcparam2=[0, 1, 0, 0])


@pytest.mark.parametrize("source,limit", [(BEAM, 256), (PLANE, 32), (SLIT, 32)], ids=["beam", "plane", "slit"])
def test_box_sums_equal_float64_sums(source, limit, monkeypatch):
    cfg = dict(nphoton=400000, vol=np.ones((40, 40, 40), np.uint8), prop=[[0, 0, 1, 1], [0.01, 1.0, 0.01, 1.37]],
               tstart=0, tend=1e-9, tstep=1e-9, isreflect=0, seed=17, mathmode=0, issavedet=1, issaveseed=1,
               savedetflag="DP", detpos=[[20, 20, 0, 12]], maxdetphoton=400000, **source)
    fwd = mcxcl_amd.run(cfg)
    n, times = 20000, 40                                    # every photon again and again: hot cells
    detp, seeds = fwd["detp"][:, :n], fwd["seeds"][:, :n]
    assert detp.shape[1] == n
    # four workgroups of 256 lanes, so that each one's box takes many photons
    rep = dict(cfg, seed=np.tile(seeds, times), detphotons=np.tile(detp, times), outputtype="jacobian", replaydet=0,
               rawfield=1, rawonly=1, issaveseed=0, autopilot=0, nthread=1024, nblocksize=64)
    monkeypatch.setenv("MCXHIP_BLOCK", "256")

    def pair(weight):
        r = dict(rep, replayweight=np.broadcast_to(np.asarray(weight, np.float32), (times * n,)).copy())
        box = mcxcl_amd.run(r)["flux64"]
        with monkeypatch.context() as m:
            m.setenv("MCXHIP_BOX_BYTES", "0")
            return box, mcxcl_amd.run(r)["flux64"]

    box, exact = pair(1.0)
    assert exact.min() >= 0 and exact.max() > 1000
    size, err = np.linalg.norm(exact), np.linalg.norm(box - exact)
    bound = 3 * 2.0 ** -24 * limit / np.sqrt(3 * exact.max() * 0.5) * size
    assert 0 < err <= bound
    for weight in (-1.0, np.where(np.arange(times * n) % 2, 1.0, -1.0)):
        box, exact = pair(weight)
        err = np.linalg.norm(box - exact)
        assert err <= bound
    box, exact = pair(1e6)
    size, err = np.linalg.norm(exact), np.linalg.norm(box - exact)
    assert err <= 2.0 ** -24 * size

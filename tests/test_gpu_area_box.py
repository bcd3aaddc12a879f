"""The deposit box under area sources: widths below, at and above what the box spans,
flat and long grids, tilted and vertical sources.  The parity build against the oracle:
energies bit-exact, the float64 grid in another order of fewer than 1e6 terms of one
sign (1e-9).  The fast build draws other photons: the absorbed weight in its grid within
six standard deviations of the oracle's, whose square is at most the weight itself (each
photon's absorbed weight lies in [0, 1])."""

import numpy as np
import pytest

import mcxcl_amd
import oracle

pytestmark = pytest.mark.gpu

_FACE = dict(srcdir=[0, 0, 1])


@pytest.mark.parametrize("dim,gates,src", [
    ((24, 24, 24), 1, dict(_FACE, srcpos=[10, 11, 0], srcparam1=[3, 0, 0, 0], srcparam2=[0, 2, 0, 0])),
    ((24, 20, 30), 3, dict(_FACE, srcpos=[2, 1, 0], srcparam1=[20, 0, 0, 0], srcparam2=[0, 18, 0, 0])),
    ((70, 66, 9), 2, dict(_FACE, srcpos=[-4, 0, -2], srcparam1=[80, 0, 0, 0], srcparam2=[0, 66, 0, 0])),
    ((120, 6, 5), 1, dict(_FACE, srcpos=[0, 2, 0], srcparam1=[120, 0, 0, 0], srcparam2=[0, 1, 0, 0])),
    ((40, 40, 40), 1, dict(_FACE, srcpos=[35, 5, 0], srcparam1=[-30, 20, 0, 0], srcparam2=[5, 10, 0, 0])),
    ((30, 40, 50), 4, dict(srcdir=[1, 0, 0], srcpos=[0, 5, 5], srcparam1=[0, 30, 0, 0], srcparam2=[0, 0, 40, 0])),
    ((30, 30, 30), 1, dict(srcdir=[0, 0.6, 0.8], srcpos=[5, 5, 15], srcparam1=[20, 0, 0, 0], srcparam2=[0, 16, -12, 0])),
])
def test_area_sources(dim, gates, src):
    cfg = dict(nphoton=20000, vol=np.ones(dim, np.uint8), prop=[[0, 0, 1, 1], [0.02, 2.0, 0.5, 1.37]], srctype="planar",
               tstart=0, tend=2e-9, tstep=2e-9 / gates, isreflect=0, seed=29, issavedet=0, **src)
    par = dict(cfg, autopilot=0, nthread=2048, nblocksize=64, mathmode=1, rawfield=1)
    gpu, ref = mcxcl_amd.run(par), oracle.run(par, nthread=2048)
    assert gpu["stat"]["energytot"] == ref["stat"]["energytot"]
    assert gpu["stat"]["energyabs"] == ref["stat"]["energyabs"]
    np.testing.assert_allclose(gpu["flux64"], ref["flux64"], rtol=1e-9, atol=1e-12)
    fast = mcxcl_amd.run(dict(cfg, mathmode=0, outputtype="energy", rawfield=1))
    esc = fast["stat"]["energytot"] - fast["stat"]["energyabs"]
    assert 0 < esc < fast["stat"]["energytot"]
    whole = oracle.run(dict(par, outputtype="energy"), nthread=2048)["flux64"].sum()
    assert abs(fast["flux64"].sum() - whole) < 6 * np.sqrt(2 * whole)     # two independent runs

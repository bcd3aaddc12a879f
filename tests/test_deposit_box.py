"""The deposit box under area sources, as the launch plan lays it out (host only): inside
the grid and the budget, over the source's middle, and no smaller than the same source's
default box where the source is narrow."""

import ctypes

import numpy as np
import pytest

from mcxcl_amd import _native, pmcxcl

BYTES = 148000     # what a 1024-lane workgroup of the default arithmetic has


def _box(dim, widths, gates=1, boxbytes=BYTES, axis=2, **over):
    """origin, edges and gates of a planar source centred on the low face of an axis"""
    a, b = (axis + 1) % 3, (axis + 2) % 3
    pos, u, v, n = np.zeros(3), np.zeros(4), np.zeros(4), np.zeros(3)
    n[axis], u[a], v[b] = 1, widths[0], widths[1]
    pos[a], pos[b] = (dim[a] - widths[0]) / 2, (dim[b] - widths[1]) / 2
    cfg = dict(nphoton=100, vol=np.ones(dim, np.uint8), prop=[[0, 0, 1, 1], [0.01, 1, 0, 1.37]], srctype="planar",
               srcpos=pos.tolist(), srcdir=n.tolist(), srcparam1=u.tolist(), srcparam2=v.tolist(), tstart=0, tend=5e-9,
               tstep=5e-9 / gates, issavedet=0, mathmode=0)
    cfg.update(over)
    with pmcxcl.prepare(cfg) as pc:
        out = (ctypes.c_uint * 7)()
        assert _native.lib.mcx_deposit_box(ctypes.byref(pc.c), boxbytes, out) == 0
    return np.array(out[:3]), np.array(out[3:6]), out[6]


@pytest.mark.parametrize("gates", [1, 2, 10])
@pytest.mark.parametrize("boxbytes", [32768, 80000, BYTES])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("dim,widths", [
    ((60, 60, 60), (40, 1)), ((60, 60, 60), (1, 40)), ((100, 100, 100), (60, 2)), ((60, 60, 60), (40, 40)),
    ((60, 60, 60), (38, 36)), ((160, 160, 160), (100, 100)), ((120, 6, 5), (120, 1)), ((9, 70, 66), (66, 70)),
    ((200, 3, 200), (3, 200)), ((256, 256, 2), (250, 3)), ((40, 41, 43), (90, 0.5)), ((64, 64, 64), (10, 5)),
])
def test_the_box_fits_and_covers(dim, widths, axis, boxbytes, gates):
    org, edge, ng = _box(dim, widths, gates, boxbytes, axis)
    assert 1 <= ng <= gates and (edge >= 1).all() and (org + edge <= dim).all()
    cells = boxbytes // 4
    assert edge.prod() * ng <= cells
    # the source's middle, on the face
    middle = np.array(dim) // 2
    middle[axis] = 0
    assert (org <= middle).all() and (middle < org + edge).all()
    # as many cells as the default box of a point there, and the slit's own flanks covered as
    # far sideways as down
    _, point, _ = _box(dim, (0, 0), gates, boxbytes, axis)
    assert edge.prod() * ng >= 0.75 * min(point.prod() * ng, np.prod(dim))
    side = [i for i in range(3) if i != axis]
    narrow = min(side, key=lambda i: edge[i])
    assert edge[narrow] >= min(edge[axis], 8, dim[narrow] - 1)


def test_square_sources_keep_their_box():
    """40x40 on 60^3 and 100x100 on 160x160x60: the shapes that were measured"""
    assert _box((60, 60, 60), (40, 40))[1].tolist() == [40, 40, 23]
    assert _box((160, 160, 60), (100, 100))[1].tolist() == [68, 68, 8]

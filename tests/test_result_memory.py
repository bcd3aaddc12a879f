"""Seeding words across the edges of the generator's runs, result arrays that take over
the library's memory, and the absorption gradient alone."""

import ctypes
import gc

import numpy as np
import pytest

import mcxcl_amd
import oracle
from mcxcl_amd import _native, pmcxcl, workloads


@pytest.mark.parametrize("n", [1, 30, 31, 34, 1023, 1024, 1025, 2048, 5000])
def test_seed_words_equal_the_c_library(n):
    got = np.zeros(n, np.uint32)
    _native.lib.mcx_host_seed_words(97, n, got.ctypes.data_as(ctypes.POINTER(ctypes.c_uint)))
    _native.libc.srand(97)
    assert got.tolist() == [_native.libc.rand() for _ in range(n)]


def test_adopted_memory_lives_with_its_last_view():
    ptr = _native.cmalloc(4 << 20)
    view = _native.adopt(ptr, ctypes.c_float, 1 << 20).reshape(1024, 1024)[5]
    view[:] = 7.0
    gc.collect()
    _native.cmalloc(4 << 20)
    assert (view == 7.0).all() and view.flags.writeable


@pytest.mark.gpu
@pytest.mark.parametrize("raw", [{}, {"rawfield": 1}, {"rawfield32": 1}, {"rawfield": 1, "rawonly": 1}])
def test_results_outlive_later_runs(raw):
    """exact: the bit-reproducible arithmetic on a fixed map, grids summed in another order
    (float64, rounded to float32: 1e-6)"""
    cfg = workloads.sphere_cube_workload(nphoton=20000, autopilot=0, nthread=2048, nblocksize=64, mathmode=1,
                                         issavedet=1, issaveseed=1, savedetflag="DSP", **raw)
    a = mcxcl_amd.run(cfg)
    kept = {k: v.copy() for k, v in a.items() if isinstance(v, np.ndarray)}
    with pmcxcl.prepare(cfg) as pc:      # a prepared run collects as often as it is asked
        if not raw:
            assert _native.lib.mcx_try_run_simulation(ctypes.byref(pc.c)) == 0
            one, two = pc.collect(), pc.collect()
            assert all(np.array_equal(one[k], two[k]) for k in kept)
    b = mcxcl_amd.run(dict(cfg, seed=1234567))
    assert all(np.array_equal(a[k], kept[k]) for k in kept)
    assert ("flux" in a) == (not raw.get("rawonly"))
    if "flux" in a:
        assert a["flux"].flags.writeable and not np.array_equal(a["flux"], b["flux"])
    if raw.get("rawfield"):
        c = mcxcl_amd.run(dict(cfg, rawonly=0))
        np.testing.assert_allclose(c["flux64"], a["flux64"], rtol=1e-9, atol=1e-12)


@pytest.mark.gpu
def test_absorption_gradient_alone_equals_the_joint_one():
    torch = pytest.importorskip("torch")
    from mcxcl_amd import autograd
    vol = np.ones((12, 10, 8), np.uint8)
    cfg = dict(nphoton=20000, vol=vol, prop=[[0, 0, 1, 1], [0.01, 1.0, 0.5, 1.37]], srcpos=[6, 5, 0], srcdir=[0, 0, 1],
               detpos=[[3, 5, 0, 2], [9, 5, 0, 2]], tstart=0, tend=1e-9, tstep=1e-9, seed=11, mathmode=1,
               autopilot=0, nthread=1024, nblocksize=64)
    grads = []
    for both in (False, True):
        mua = torch.full(vol.shape, 0.01, requires_grad=True)
        mus = torch.full(vol.shape, 1.0, requires_grad=both)
        autograd.detector_signals(mua, mus, cfg).sum().backward()
        assert (mus.grad is not None) == both
        grads.append(mua.grad.numpy())
    # the replay's float64 deposits in another order, rounded to float32
    np.testing.assert_allclose(grads[0], grads[1], rtol=1e-6, atol=1e-12)
    assert np.abs(grads[0]).sum() > 0


@pytest.mark.parametrize("scratch", [0, 10, 500])
def test_hand_over_slots_stay_within_their_bound(scratch):
    """the default map has them, and no map takes more than 1 GiB for them"""
    words = _native.lib.mcx_hand_over_words
    assert words(655360 // 256, 256, scratch) == 655360 // 4 * (42 + scratch)
    assert words(256, 1024, scratch) == 65536 * (42 + scratch) and words(40000, 64, scratch) == 0
    for lanes in (1 << 20, 1 << 22, 10 ** 7, 1 << 26, 1 << 30):
        assert 4 * words(lanes // 256, 256, scratch) <= 1 << 30


@pytest.mark.parametrize("tend,tstep", [(3e-10, 2e-10), (5e-10, 2e-10), (1e-9, 4e-10), (1.3e-9, 2e-10), (5e-9, 5e-10),
                                        (5e-9, 1.1e-9)])
def test_gates_are_counted_as_the_library_does(tend, tstep):
    """windows of a whole number of gates and a half, where single and double precision round
    to different counts: the arrays handed to the library hold what it fills"""
    cfg = workloads.homogeneous_cube_workload(nphoton=100, vol=np.ones((5, 6, 7), np.uint8), srcpos=[2, 2, 0],
                                              tstart=0, tend=tend, tstep=tstep)
    out = oracle.run(dict(cfg, autopilot=0, nthread=64, nblocksize=64), nthread=64)
    with pmcxcl.prepare(dict(cfg, rawfield=1)) as pc:
        assert pc.raw.size == out["flux64"].size
    assert out["flux"].shape[3] == out["flux64"].shape[3]


@pytest.mark.gpu
@pytest.mark.parametrize("extra", [{}, {"omega": 2 * np.pi * 1e8}, {"tstep": 5e-10}])
def test_returned_field_holds_no_more_than_itself(extra):
    """the array that is handed over keeps the block it was read back into: the field's size,
    up to the allocator's rounding"""
    _native.libc.malloc_usable_size.restype = ctypes.c_size_t
    _native.libc.malloc_usable_size.argtypes = [ctypes.c_void_p]
    cfg = dict(workloads.sphere_cube_workload(nphoton=2000, issavedet=0), **extra)
    with pmcxcl.prepare(cfg) as pc:
        assert _native.lib.mcx_try_run_simulation(ctypes.byref(pc.c)) == 0
        assert _native.libc.malloc_usable_size(pc.c.exportfield) <= 4 * pc.fieldlen + 8192

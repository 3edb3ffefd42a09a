"""GPU parity of the 3D plane passes where they run in chunks on two streams
(W2 larger than two chunks of 96 MB): FP64 tendencies and CFL maxima of ns3d
and ns3d.strat on a grid of a few unequal chunks against the FP64 oracle
(relative L2 1e-12, the bar of the other tendency tests), and the fused
stages captured in a HIP graph against the eager ones, bit for bit, over
several replays with eager work between them.
"""

import ctypes

import numpy as np
import pytest

from fluidsim_amd import _lib
from fluidsim_amd.synthetic import ns3d_spectrum_vv_fft
from oracle.operators import Oper3D
from oracle.solvers import NS3D, NS3DStrat

from .gpu_helpers import host, make_plan, rel_l2, to_dev_complex, torch, zeros_complex

pytestmark = pytest.mark.gpu

NX, NY, NZ = 256, 256, 102  # W2 in FP64: 220 MB (ns3d), 257 MB (strat); 25 or 26 planes a chunk


def _case(strat, shape=(NX, NY, NZ)):
    oper = Oper3D(*shape)
    vv = ns3d_spectrum_vv_fft(*shape, seed=3)
    if strat:
        sim = NS3DStrat(oper, N=4.0)
        sim.init_from_fft(*vv, 0.5 * vv[0])
    else:
        sim = NS3D(oper)
        sim.init_from_vxvyvzfft(*vv)
    return sim


@pytest.mark.parametrize("strat", [False, True])
def test_chunked_tendency(strat):
    print(f"case chunked planes strat={strat}", flush=True)
    sim = _case(strat)
    ref = sim.tendencies_nonlin(sim.state_spect)
    plan = make_plan(sim.oper, 8, 7)
    S = to_dev_complex(sim.state_spect, 8)
    out = zeros_complex(S.shape, 8)
    s = _lib.stream_ptr()
    _lib.call("fsx_reset_maxima", plan.handle, s)
    if strat:
        _lib.call("fsx_strat_tendency", plan.handle, _lib.dptr(S), _lib.dptr(out), 0, 0.0, 4.0,
                  1, 0, 1, s)
    else:
        _lib.call("fsx_ns3d_tendency", plan.handle, _lib.dptr(S), _lib.dptr(out), 0, 0.0, 1, s)
        _lib.call("fsx_project", plan.handle, *(_lib.dptr(out[i]) for i in range(3)), 1, s)
    assert rel_l2(host(out), ref) < 1e-12
    sc = (ctypes.c_double * 6)()
    _lib.call("fsx_get_scalars", plan.handle, sc, s)
    for i in range(3):
        v = sim.oper.ifft(sim.state_spect[i])
        assert sc[i] == pytest.approx(np.abs(v).max(), rel=1e-12)


def test_chunked_stages_in_a_graph():
    t = torch()
    sim = _case(False)
    plan = make_plan(sim.oper, 8, 6)
    S0 = to_dev_complex(sim.state_spect, 8)
    stream = t.cuda.Stream()
    sp = _lib.stream_ptr(stream)
    _lib.call("fsx_set_dt", plan.handle, 1e-3, sp)
    vc = _lib.doubles([1e-3, 0, 0, 0])

    def buffers():
        return S0.clone(), t.zeros_like(S0), t.zeros_like(S0)

    def step(S, tmp, t1):
        for stage in range(4):
            _lib.call("fsx_ns3d_rk_stage", plan.handle, 4, stage, _lib.dptr(S), _lib.dptr(tmp),
                      _lib.dptr(t1), 0, 0.0, 1, 0, vc, 0.5, 0.2, sp)

    eager, graph = buffers(), buffers()
    t.cuda.synchronize()
    step(*eager)
    h = ctypes.c_void_p()
    _lib.call("fsx_graph_begin", sp)
    try:
        step(*graph)
    finally:
        rc = _lib.get_lib().fsx_graph_end(sp, ctypes.byref(h))
    _lib.check(rc, "fsx_graph_end")
    for i in range(3):
        if i:
            step(*eager)
        _lib.call("fsx_graph_launch", h, sp)
        stream.synchronize()
        assert t.equal(eager[0], graph[0]), f"replay {i}"
    _lib.call("fsx_graph_destroy", h)


# FP64 on ragged axes (mixed-radix rows of even and odd length, W2 211 MB) and
# FP32 (215 MB; LDS rows of 640 points, register rows of 256), chunks of unequal
# size; FP32: eps log2 of the points is 1.4e-6, with a factor of 3
@pytest.mark.parametrize("strat", [False, True])
@pytest.mark.parametrize("shape, prec, tol", [((240, 192, 143), 8, 1e-12),
                                              ((189, 250, 134), 8, 1e-12),
                                              ((256, 256, 182), 4, 4e-6),
                                              ((640, 96, 202), 4, 4e-6)])
def test_chunked_tendency_of_other_rows(strat, shape, prec, tol):
    print(f"case chunked planes {shape} strat={strat} prec={prec}", flush=True)
    sim = _case(strat, shape)
    ref = sim.tendencies_nonlin(sim.state_spect)
    plan = make_plan(sim.oper, prec, 7)
    S = to_dev_complex(sim.state_spect, prec)
    out = zeros_complex(S.shape, prec)
    s = _lib.stream_ptr()
    _lib.call("fsx_reset_maxima", plan.handle, s)
    _lib.call("fsx_timing_enable", plan.handle, 1)
    if strat:
        _lib.call("fsx_strat_tendency", plan.handle, _lib.dptr(S), _lib.dptr(out), 0, 0.0, 4.0,
                  1, 0, 1, s)
    else:
        _lib.call("fsx_ns3d_tendency", plan.handle, _lib.dptr(S), _lib.dptr(out), 0, 0.0, 1, s)
        _lib.call("fsx_project", plan.handle, *(_lib.dptr(out[i]) for i in range(3)), 1, s)
    ms, by, cn = ctypes.c_double(), ctypes.c_double(), ctypes.c_longlong()
    _lib.call("fsx_timing_read_planes", plan.handle, ctypes.byref(ms), ctypes.byref(by),
              ctypes.byref(cn), 1)
    _lib.call("fsx_timing_enable", plan.handle, 0)
    assert cn.value == 1  # it did run in chunks
    assert rel_l2(host(out), ref) < tol
    sc = (ctypes.c_double * 6)()
    _lib.call("fsx_get_scalars", plan.handle, sc, s)
    for i in range(3):
        v = sim.oper.ifft(sim.state_spect[i])
        assert sc[i] == pytest.approx(np.abs(v).max(), rel=tol)


def test_chunked_strat_stages_in_a_graph():
    """As test_chunked_stages_in_a_graph, for ns3d.strat."""
    t = torch()
    sim = _case(True)
    plan = make_plan(sim.oper, 8, 7)
    S0 = to_dev_complex(sim.state_spect, 8)
    stream = t.cuda.Stream()
    sp = _lib.stream_ptr(stream)
    _lib.call("fsx_set_dt", plan.handle, 1e-3, sp)
    vc = _lib.doubles([1e-3, 0, 0, 0])
    eager, graph = ((S0.clone(), t.zeros_like(S0), t.zeros_like(S0)) for _ in range(2))

    def step(bufs):
        for stage in range(4):
            _lib.call("fsx_strat_rk_stage", plan.handle, 4, stage, *map(_lib.dptr, bufs), 0, 0.0,
                      4.0, 1, 0, vc, 0.5, 0.2, sp)

    t.cuda.synchronize()
    step(eager)
    h = ctypes.c_void_p()
    _lib.call("fsx_graph_begin", sp)
    try:
        step(graph)
    finally:
        rc = _lib.get_lib().fsx_graph_end(sp, ctypes.byref(h))
    _lib.check(rc, "fsx_graph_end")
    for i in range(3):
        if i:
            step(eager)
        _lib.call("fsx_graph_launch", h, sp)
        stream.synchronize()
        assert t.equal(eager[0], graph[0]), f"replay {i}"
    _lib.call("fsx_graph_destroy", h)


@pytest.mark.parametrize("strat", [False, True])
def test_timing_of_overlapped_passes(strat):
    """The plane passes are timed as one block per stage with the bytes of
    the three passes, the times of all kinds fit into the time of the steps,
    and a second read after a reset holds nothing."""
    t = torch()
    sim = _case(strat)
    plan = make_plan(sim.oper, 8, 7)
    S = to_dev_complex(sim.state_spect, 8)
    tmp, t1 = t.zeros_like(S), t.zeros_like(S)
    s = _lib.stream_ptr()
    _lib.call("fsx_set_dt", plan.handle, 1e-3, s)
    vc = _lib.doubles([1e-3, 0, 0, 0])

    def step():
        for stage in range(4):
            bufs = (plan.handle, 4, stage, _lib.dptr(S), _lib.dptr(tmp), _lib.dptr(t1), 0, 0.0)
            if strat:
                _lib.call("fsx_strat_rk_stage", *bufs, 4.0, 1, 0, vc, 0.5, 0.2, s)
            else:
                _lib.call("fsx_ns3d_rk_stage", *bufs, 1, 0, vc, 0.5, 0.2, s)

    def read():
        ms, by, cn = ctypes.c_double(), ctypes.c_double(), ctypes.c_longlong()
        _lib.call("fsx_timing_read_planes", plan.handle, ctypes.byref(ms), ctypes.byref(by),
                  ctypes.byref(cn), 0)
        kinds = (ctypes.c_double * 8)(), (ctypes.c_double * 8)(), (ctypes.c_longlong * 8)()
        _lib.call("fsx_timing_read", plan.handle, *kinds, 1)
        return ms.value, by.value, cn.value, kinds

    step()
    _lib.call("fsx_timing_enable", plan.handle, 1)
    e0, e1 = t.cuda.Event(enable_timing=True), t.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(3):
        step()
    e1.record()
    ms, by, cn, (ms8, by8, cn8) = read()
    e1.synchronize()
    assert cn == 12 and list(cn8[1:4]) == [0, 0, 0] and cn8[0] == 12 and cn8[4] == 12
    kept = sim.oper.where_dealiased == 0
    mx, nyk = kept.any((0, 1)).sum(), kept.any((0, 2)).sum()
    nin, nout = (7, 6) if strat else (6, 3)
    assert by == 12 * 16 * NZ * mx * (nin + nout) * (nyk + 2 * NY)
    assert 0 < ms and ms + sum(ms8) <= e0.elapsed_time(e1)
    ms, by, cn, (ms8, by8, cn8) = read()
    assert ms == by == cn == 0 and sum(ms8) == sum(cn8) == 0
    _lib.call("fsx_timing_enable", plan.handle, 0)

"""GPU parity of the passes along axes of 2 to 16 points (thin slabs, very
small boxes), whose transforms fit a thread, and of the small problems whose
passes give a thread fewer elements, at few lines and at more than one
workgroup of them, against the FP64 oracle.

Tolerance: rounding grows like eps log2 N (eps 1.1e-16 / 6e-8) over the passes
of a step of up to 256 x 16 x 256 points: 1e-13 (FP64) and 4e-6 (FP32)
relative L2 leave a factor of 20.
"""

import numpy as np
import pytest

from fluidsim_amd import _lib
from fluidsim_amd.synthetic import ns2d_noise_rot_fft, ns3d_spectrum_vv_fft
from oracle.operators import Oper2D, Oper3D
from oracle.solvers import NS2D, NS3D, NS3DStrat

from .gpu_helpers import (host, make_plan, rel_l2, to_dev_complex, to_dev_real, zeros_complex,
                          zeros_real)

pytestmark = pytest.mark.gpu

TOL = {8: 1e-13, 4: 4e-6}


def _step(plan, S0, prec, name, args):
    S = to_dev_complex(S0, prec)
    tmp, t1 = zeros_complex(S.shape, prec), zeros_complex(S.shape, prec)
    s = _lib.stream_ptr()
    _lib.call("fsx_set_dt", plan.handle, 0.01, s)
    for stage in range(4):
        _lib.call(name, plan.handle, 4, stage, _lib.dptr(S), _lib.dptr(tmp), _lib.dptr(t1), *args,
                  _lib.doubles([1e-3, 0, 0, 0]), 0.0, 0.2, s)
    return host(S)


@pytest.mark.parametrize("prec", [8, 4])
@pytest.mark.parametrize("n", [2, 4, 8, 16])
@pytest.mark.parametrize("nx, other", [(6, 4), (200, 3), (34, 70)])
def test_transforms(n, nx, other, prec):
    print(f"case short axes transforms n={n} nx={nx} other={other} prec={prec}", flush=True)
    rng = np.random.default_rng(n)
    opers = [Oper2D(nx, n, 2 * np.pi, 3.0), Oper3D(nx, n, other, 2 * np.pi, 3.0, 1.0),
             Oper3D(nx, other, n, 2 * np.pi, 3.0, 1.0), Oper3D(nx, n, n, 2 * np.pi, 3.0, 1.0)]
    for oper in opers:
        x = rng.standard_normal((2,) + oper.shapeX)
        plan = make_plan(oper, prec, 1, dealias=False)
        k = zeros_complex((2,) + oper.shapeK, prec)
        xd = to_dev_real(x, prec)
        _lib.call("fsx_fft", plan.handle, _lib.dptr(xd), _lib.dptr(k), 2, _lib.stream_ptr())
        assert rel_l2(host(k), np.array([oper.fft(a) for a in x])) < TOL[prec]
        back = zeros_real((2,) + oper.shapeX, prec)
        _lib.call("fsx_ifft", plan.handle, _lib.dptr(k), _lib.dptr(back), 2, _lib.stream_ptr())
        assert rel_l2(host(back), x) < TOL[prec]


@pytest.mark.parametrize("prec", [8, 4])
@pytest.mark.parametrize("nx, ny", [(16, 2), (300, 4), (16, 8), (16, 16), (300, 16), (32, 32),
                                    (128, 64), (64, 128), (300, 256), (96, 512), (40, 1024)])
def test_ns2d_step(nx, ny, prec):
    print(f"case small ns2d step {nx} x {ny} prec={prec}", flush=True)
    sim = NS2D(Oper2D(nx, ny), nu_2=1e-3)
    sim.init_from_rotfft(ns2d_noise_rot_fft(nx, ny, seed=ny, kmax=4))
    S0 = sim.state_spect.copy()
    sim.run_with_dts([0.01])
    out = _step(make_plan(sim.oper, prec, 4), S0, prec, "fsx_ns2d_rk_stage", (0.0,))
    assert rel_l2(out, sim.state_spect) < TOL[prec]


@pytest.mark.parametrize("prec", [8, 4])
@pytest.mark.parametrize("strat", [False, True])
@pytest.mark.parametrize("shape", [(16, 16, 16), (32, 16, 2), (34, 70, 4), (256, 20, 8),
                                   (256, 16, 16), (20, 4, 64), (64, 32, 32), (24, 128, 64),
                                   (20, 16, 256)])
def test_3d_step(shape, strat, prec):
    print(f"case small 3D step {shape} strat={strat} prec={prec}", flush=True)
    oper = Oper3D(*shape)
    vv = ns3d_spectrum_vv_fft(*shape, seed=7)
    if strat:
        sim = NS3DStrat(oper, N=4.0, nu_2=1e-3)
        sim.init_from_fft(*vv, 0.5 * vv[0])
    else:
        sim = NS3D(oper, nu_2=1e-3)
        sim.init_from_vxvyvzfft(*vv)
    S0 = sim.state_spect.copy()
    sim.run_with_dts([0.01])
    name = "fsx_strat_rk_stage" if strat else "fsx_ns3d_rk_stage"
    args = (0, 0.0, 4.0, 1, 0) if strat else (0, 0.0, 1, 0)
    out = _step(make_plan(oper, prec, 7), S0, prec, name, args)
    assert rel_l2(out, sim.state_spect) < TOL[prec]


@pytest.mark.parametrize("prec", [8, 4])
@pytest.mark.parametrize("n", [512, 1024])
def test_tile_settings_give_the_same_bits_at_the_small_problem_limit(n, prec):
    """The elements per thread of a pass do not depend on the tile settings:
    one output field per workgroup (four times the waves) or all four, any lines
    per tile, at sizes on both sides of the small-problem limit."""
    print(f"case tile settings n={n} prec={prec}", flush=True)
    oper = Oper2D(n, n)
    plan = make_plan(oper, prec, 4)
    rot = to_dev_complex(ns2d_noise_rot_fft(n, n, seed=n, kmax=12), prec)
    outs = []
    for split, inv, fwd in ((0, 0, 0), (1, 0, 0), (1, 2, 1), (0, 8, 4)):
        _lib.call("fsx_plan_set_tiles", plan.handle, inv, fwd, split)
        out = zeros_complex(oper.shapeK, prec)
        _lib.call("fsx_ns2d_tendency", plan.handle, _lib.dptr(rot), _lib.dptr(out), 0.0, 0,
                  _lib.stream_ptr())
        outs.append(host(out))
    for o in outs[1:]:
        assert np.array_equal(o, outs[0])

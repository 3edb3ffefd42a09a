"""GPU parity of the strided (y and z) passes at every power-of-two length
they have a plan for, at the edges of their tiles, against the FP64 oracle.

One Runge-Kutta step of each solver through the fused stages runs every
strided pass of the solver.  Tolerance: the passes are FFTs of length N with
a few operations per point around them, whose rounding error grows like
eps log2 N (eps 1.1e-16 / 6e-8): 1e-13 (FP64) and 4e-6 (FP32) relative L2
leave a factor of 20 at N = 8192.
"""

import numpy as np
import pytest

from fluidsim_amd import _lib
from fluidsim_amd.synthetic import ns2d_noise_rot_fft, ns3d_spectrum_vv_fft
from oracle.operators import Oper2D, Oper3D
from oracle.solvers import NS2D, NS3D, NS3DStrat

from .gpu_helpers import host, make_plan, rel_l2, to_dev_complex, zeros_complex

pytestmark = pytest.mark.gpu

TOL = {8: 1e-13, 4: 4e-6}


def _fused_step(plan, S0, prec, dt, visc, call, nstages=4):
    S = to_dev_complex(S0, prec)
    tmp, t1 = zeros_complex(S.shape, prec), zeros_complex(S.shape, prec)
    s = _lib.stream_ptr()
    _lib.call("fsx_set_dt", plan.handle, float(dt), s)
    vc = _lib.doubles(visc)
    for stage in range(nstages):
        call(plan.handle, stage, _lib.dptr(S), _lib.dptr(tmp), _lib.dptr(t1), vc, s)
    return host(S)


def _ns2d(h, stage, S, tmp, t1, vc, s):
    _lib.call("fsx_ns2d_rk_stage", h, 4, stage, S, tmp, t1, 0.0, vc, 0.0, 0.2, s)


def _ns3d(h, stage, S, tmp, t1, vc, s):
    _lib.call("fsx_ns3d_rk_stage", h, 4, stage, S, tmp, t1, 0, 0.0, 1, 0, vc, 0.0, 0.2, s)


def _strat(h, stage, S, tmp, t1, vc, s):
    _lib.call("fsx_strat_rk_stage", h, 4, stage, S, tmp, t1, 0, 0.0, 4.0, 1, 0, vc, 0.0, 0.2, s)


# nx: 6 kept kx (a tile wider than the pass) and 43 (ragged last tile)
@pytest.mark.parametrize("nx", [16, 128])
@pytest.mark.parametrize("prec", [8, 4])
@pytest.mark.parametrize("ny", [32, 64, 128, 256, 512, 1024, 2048, 4096, 8192])
def test_ns2d_step(ny, prec, nx):
    if ny == 8192 and (prec == 8 or nx > 16):
        pytest.skip("longer than an FP64 tile; one FP32 case is enough")
    print(f"case ns2d step ny={ny} nx={nx} prec={prec}", flush=True)
    sim = NS2D(Oper2D(nx, ny), nu_2=1e-3)
    sim.init_from_rotfft(ns2d_noise_rot_fft(nx, ny, seed=ny, kmax=4))
    S0 = sim.state_spect.copy()
    sim.run_with_dts([0.01])
    out = _fused_step(make_plan(sim.oper, prec, 4), S0, prec, 0.01, [1e-3, 0, 0, 0], _ns2d)
    assert rel_l2(out, sim.state_spect) < TOL[prec]


@pytest.mark.parametrize("prec", [8, 4])
@pytest.mark.parametrize("strat", [False, True])
@pytest.mark.parametrize("nz", [32, 64, 128, 256, 512, 1024, 2048, 4096])
def test_3d_step(nz, strat, prec):
    print(f"case 3D step nz={nz} strat={strat} prec={prec}", flush=True)
    nx, ny = 34, 32
    oper = Oper3D(nx, ny, nz)
    vv = ns3d_spectrum_vv_fft(nx, ny, nz, seed=nz)
    if strat:
        sim = NS3DStrat(oper, N=4.0, nu_2=1e-3)
        sim.init_from_fft(*vv, 0.5 * vv[0])
    else:
        sim = NS3D(oper, nu_2=1e-3)
        sim.init_from_vxvyvzfft(*vv)
    S0 = sim.state_spect.copy()
    sim.run_with_dts([0.01])
    out = _fused_step(make_plan(oper, prec, 7), S0, prec, 0.01, [1e-3, 0, 0, 0],
                      _strat if strat else _ns3d)
    assert rel_l2(out, sim.state_spect) < TOL[prec]


def test_axis_with_nyquist_kept_and_a_gap():
    """A mask that keeps the Nyquist index of y and prunes part of the
    negative ones (no truncation of the solvers does) is pruned by the mask."""
    n = 64
    oper = Oper2D(n, n)
    mask = oper.where_dealiased.copy()
    mask[n // 2, :5] = 0
    oper.where_dealiased = mask
    sim = NS2D(oper, nu_2=1e-3)
    sim.init_from_rotfft(ns2d_noise_rot_fft(n, n, seed=1))
    S0 = sim.state_spect.copy()
    sim.run_with_dts([0.01])
    out = _fused_step(make_plan(oper, 8, 4), S0, 8, 0.01, [1e-3, 0, 0, 0], _ns2d)
    assert rel_l2(out, sim.state_spect) < TOL[8]

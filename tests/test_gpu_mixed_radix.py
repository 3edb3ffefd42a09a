"""GPU parity of the mixed-radix passes (lengths that are not powers of two)
with numpy and the FP64 oracle, at lengths that take every butterfly (2 to
13, 15, 16, other primes by the direct DFT) as the only and as a later stage,
in one LDS buffer and in two, for even and odd row lengths.

Tolerances: rounding grows like eps log N in the butterflies and like eps N
in a direct DFT of a prime N; 1e-13 (FP64) and 4e-6 (FP32) relative L2 leave a
factor of 10 at the largest prime here (89).
"""

import numpy as np
import pytest

from fluidsim_amd import _lib
from fluidsim_amd.synthetic import ns2d_noise_rot_fft
from oracle.operators import Oper2D
from oracle.solvers import NS2D

from .gpu_helpers import (host, make_plan, rel_l2, to_dev_complex, to_dev_real, zeros_complex,
                          zeros_real)

pytestmark = pytest.mark.gpu

TOL = {8: 1e-13, 4: 4e-6}

# 2 stages of every pair class, 3 and 4 stages, direct primes (17, 23, 29, 89),
# more values per tile than registers (2047 = 23 89, 1998 = 2 27 37)
LENGTHS = [2, 3, 5, 6, 7, 9, 10, 11, 12, 13, 15, 17, 21, 26, 28, 33, 45, 48, 54, 58, 77, 90, 99,
           100, 105, 117, 121, 130, 143, 150, 169, 180, 195, 210, 225, 240, 364, 495, 675, 1001,
           1155, 1998, 2047]


@pytest.mark.parametrize("prec", [8, 4])
@pytest.mark.parametrize("n", LENGTHS)
def test_transforms(n, prec):
    print(f"case mixed radix transforms n={n} prec={prec}", flush=True)
    rng = np.random.default_rng(n)
    for nx, ny in ((n, 6), (12, n)):  # as the row length, as the strided length
        oper = Oper2D(nx, ny, 2 * np.pi, 3.0)
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
@pytest.mark.parametrize("shape", [(48, 48), (45, 50), (99, 36), (130, 105), (240, 77),
                                   (58, 169), (1001, 24), (24, 1155)])
def test_ns2d_step(shape, prec):
    """The products between the transforms (rows of even and odd length) and
    the fused Runge-Kutta stages."""
    print(f"case mixed radix ns2d step {shape} prec={prec}", flush=True)
    nx, ny = shape
    sim = NS2D(Oper2D(nx, ny), nu_2=1e-3)
    sim.init_from_rotfft(ns2d_noise_rot_fft(nx, ny, seed=nx, kmax=6))
    S = to_dev_complex(sim.state_spect, prec)
    sim.run_with_dts([0.01])
    plan = make_plan(sim.oper, prec, 4)
    tmp, t1 = zeros_complex(S.shape, prec), zeros_complex(S.shape, prec)
    s = _lib.stream_ptr()
    _lib.call("fsx_set_dt", plan.handle, 0.01, s)
    vc = _lib.doubles([1e-3, 0, 0, 0])
    for stage in range(4):
        _lib.call("fsx_ns2d_rk_stage", plan.handle, 4, stage, _lib.dptr(S), _lib.dptr(tmp),
                  _lib.dptr(t1), 0.0, vc, 0.0, 0.2, s)
    assert rel_l2(host(S), sim.state_spect) < TOL[prec]

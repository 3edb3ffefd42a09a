"""Transforms of a flat FP64 grid whose z-passes reach far: 4096 x 4096 x 128,
one field of 17 GB, neighbouring z positions 134 MB apart.  A few plane waves,
at z wavenumbers (and so output positions) all over the axis, against their
closed form, and every other mode against zero.

Tolerance: eps log2(2^31 points) with a factor of 30: 1e-13 of the largest
amplitude.
"""

import numpy as np
import pytest

from fluidsim_amd import _lib

from .gpu_helpers import torch

pytestmark = pytest.mark.gpu

NX, NY, NZ = 4096, 4096, 128
# (kx, ky, kz): amplitude; kx in 1 .. nx / 2 - 1, so that one mode of the half
# spectrum is one wave
MODES = {(1, 0, 30): 1.0 - 0.5j, (2047, -2047, 31): 0.25 + 1.0j, (700, 2047, -34): -0.75j,
         (3, -1, -33): 0.5 + 0.5j, (64, 31, -2): 1.0, (1500, 1024, -1): -0.25 + 0.5j,
         (9, 5, 0): 0.125, (77, -300, 62): 1.0j, (5, 5, 95 - NZ): 0.75}


def _plane(t, z):
    """Plane z of the sum of the waves 2 Re(a exp(i k x))."""
    def wave(k, n):
        a = 2 * np.pi * ((k * np.arange(n)) % n) / n
        return t.from_numpy(np.exp(1j * a)).cuda()

    x = t.zeros((NY, NX), dtype=t.float64, device="cuda")
    for (kx, ky, kz), a in MODES.items():
        az = 2 * a * np.exp(2j * np.pi * ((kz * z) % NZ) / NZ)
        ey, ex = az * wave(ky, NY), wave(kx, NX)
        x += t.outer(ey.real, ex.real) - t.outer(ey.imag, ex.imag)
    return x


def test_transforms_of_a_flat_grid():
    t = torch()
    free, _ = t.cuda.mem_get_info()
    if free < 80e9:
        pytest.skip("needs 80 GB of free device memory")
    print(f"case transforms {NX} x {NY} x {NZ} float64", flush=True)
    plan = _lib.Plan(3, NX, NY, NZ, 2 * np.pi, 2 * np.pi, 1.0, 8, None, 1)
    x = t.empty((NZ, NY, NX), dtype=t.float64, device="cuda")
    for z in range(NZ):
        x[z] = _plane(t, z)
    k = t.empty((NZ, NY, NX // 2 + 1), dtype=t.complex128, device="cuda")
    k.fill_(float("nan"))
    _lib.call("fsx_fft", plan.handle, _lib.dptr(x), _lib.dptr(k), 1, _lib.stream_ptr())
    for (kx, ky, kz), a in MODES.items():
        got = complex(k[kz, ky, kx])
        assert abs(got - a) < 1e-13, (kx, ky, kz, got)
        k[kz, ky, kx] = 0
    rest = [float(t.view_as_real(k[z]).abs().max()) for z in range(NZ)]
    assert max(rest) < 1e-13 and not np.isnan(rest).any(), np.argmax(rest)

    k.zero_()
    for (kx, ky, kz), a in MODES.items():
        k[kz, ky, kx] = a
    x.fill_(float("nan"))
    _lib.call("fsx_ifft", plan.handle, _lib.dptr(k), _lib.dptr(x), 1, _lib.stream_ptr())
    err = [float((x[z] - _plane(t, z)).abs().max()) for z in range(NZ)]
    assert max(err) < 1e-12 and not np.isnan(err).any(), np.argmax(err)
    del x, k, plan
    t.cuda.empty_cache()

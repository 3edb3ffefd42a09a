"""Spectra of rows long enough for the transposed kx histogram (256 bins and
more): every histogram in one pass against the histograms taken one at a
time, where the kx one is not transposed, and against NumPy.

Bar: FP64 sums of a few thousand terms of one sign, and for the shares of
neighbouring bins |k| / dk to a few units in its last place (|k| / dk < 600):
1e-12 of the largest value.
"""

import numpy as np
import pytest
import torch

from fluidsim_amd.base import diagnostics as G
from fluidsim_amd.solvers.ns3d.solver import Simul

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [508, 510, 512, 514, 1020, 1026])
@pytest.mark.parametrize("precision", ["float32", "float64"])
def test_spectra_of_long_rows(nx, precision):
    params = Simul.create_default_params()
    params.oper.nx, params.oper.ny, params.oper.nz = nx, 12, 8
    params.oper.Lx, params.oper.Ly, params.oper.Lz = 7.0, 5.0, 6.0
    params.oper.precision = precision
    params.output.HAS_TO_SAVE = False
    oper = Simul(params).oper
    nkx = nx // 2 + 1
    rng = np.random.default_rng(nx)
    f = rng.standard_normal((3, 8, 12, nkx)) + 1j * rng.standard_normal((3, 8, 12, nkx))
    f = f.astype(np.complex64 if precision == "float32" else np.complex128)
    fields = [torch.from_numpy(a.copy()).cuda() for a in f]
    flags = G.KX | G.KY | G.KZ | G.SHELL | G.KZKH
    got = G.run(oper, G.NS3D_SPECTRA, flags, fields)
    for flag, key in ((G.KX, "kx"), (G.KY, "ky"), (G.KZ, "kz"), (G.SHELL, "shell"),
                      (G.KZKH, "kzkh")):
        alone = G.run(oper, G.NS3D_SPECTRA, flag, fields)[key]
        assert np.abs(got[key] - alone).max() <= 1e-12 * np.abs(alone).max(), key
    w = np.full(nkx, 2.0)
    w[0] = 1.0
    if nx % 2 == 0:
        w[-1] = 1.0
    e = 0.5 * np.abs(f.astype(np.complex128)) ** 2 * w
    dk = [2 * np.pi / L for L in (7.0, 5.0, 6.0)]
    ref = e.sum((1, 2)) / dk[0]
    assert np.abs(got["kx"][:3] - ref).max() <= 1e-12 * ref.max()
    ky = np.fft.fftfreq(12, 1 / 12) * dk[1]
    kz = np.fft.fftfreq(8, 1 / 8) * dk[2]
    k = np.sqrt((np.arange(nkx) * dk[0]) ** 2 + ky[:, None] ** 2 + kz[:, None, None] ** 2)
    n = got["shell"].shape[1]
    j = np.minimum((k / max(dk)).astype(int), n - 1)
    c = np.where(j < n - 1, k / max(dk) - j, 0.0)
    for q in range(3):
        ref = (np.bincount(j.ravel(), (e[q] * (1 - c)).ravel(), n + 1)
               + np.bincount(j.ravel() + 1, (e[q] * c).ravel(), n + 1))[:n] / max(dk)
        assert np.abs(got["shell"][q] - ref).max() <= 1e-12 * ref.max()

"""The observables and density extracts against the oracle where their kernels'
tiles end: one tile per axis, walks of x that the plane count does not divide,
rows shorter than a wavefront, the longest rows, and a field that is O(1) on
every face (the derivatives' boundary rules and the end weights count)."""
import numpy as np
import pytest

import dbecpy
from conftest import params, rel

pytestmark = pytest.mark.gpu

TOL = 1e-12  # sums of up to 1e6 terms of one sign: about 1e-15, and the bar of the single operators


@pytest.mark.parametrize("mode", [dbecpy.IMAG, dbecpy.REAL], ids=["imag", "real"])
@pytest.mark.parametrize("n", [(16, 16, 16), (80, 16, 48), (16, 32, 512), (512, 16, 16), (48, 320, 32), (160, 64, 96)],
                         ids=lambda n: "x".join(map(str, n)))
def test_observables_at_tile_edges(hip_lib, oracle_lib, mode, n):
    print(f"[gpu-case] observables mode={mode} grid={n}", flush=True)
    p = params(n=n, h=tuple(6.0 / k for k in n), dt=0.002, cutoff=2.5)
    x, y, z = dbecpy.grid(p)
    X, Y, Z = np.meshgrid(x, y, z, indexing="ij")
    f = 1.0 + 0.4 * np.cos(0.7 * X + 0.3 * Y) * np.sin(0.5 * Z + 0.2) + 0.1 * X
    if mode == dbecpy.REAL:
        f = f * np.exp(1j * (0.9 * X - 0.6 * Z + 0.4 * Y))
    with dbecpy.Solver(hip_lib, p, mode) as g, dbecpy.Solver(oracle_lib, p, mode) as o, \
            dbecpy.Solver(hip_lib, p, mode, dbecpy.MIXED) as m, dbecpy.Solver(oracle_lib, p, mode) as o32:
        f32 = f.astype(np.complex64 if mode == dbecpy.REAL else np.float32).astype(f.dtype)
        for s, psi in ((g, f), (o, f), (m, f32), (o32, f32)):
            s.set_psi(psi)
            s.set_coupling(60.0, 0.0)  # no dipolar term: the mixed form's phi is FP32
        for a, b in ((g, o), (m, o32)):
            assert a.calcnorm() == pytest.approx(b.calcnorm(), rel=TOL)
            assert a.calcmuen() == pytest.approx(b.calcmuen(), rel=TOL)
            assert a.calcmuen_phase() == pytest.approx(b.calcmuen_phase(), rel=TOL)
            assert a.calcrms() == pytest.approx(b.calcrms(), rel=TOL)
            assert a.psi_center() == pytest.approx(b.psi_center(), rel=TOL)
            for kind in range(10):
                for o3 in ((1, 1, 1), (3, 2, 5), (1000, 7, 1)):
                    u, v = a.density(kind, *o3), b.density(kind, *o3)
                    assert u.shape == v.shape
                    assert rel(u, v) < TOL, (kind, o3)

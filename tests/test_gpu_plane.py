"""The plane kernels (whole (y, z) planes in LDS: y and z sweeps with the next
forward z and y passes, inverse y and z passes with calcnu) against the oracle:
every pair of plane lengths they take, and the plane counts at which the
inverse kernel shares a plane among workgroups, adds workgroups for the last
plane or takes a second round for it."""
import numpy as np
import pytest

import dbecpy
from conftest import params, rel

pytestmark = pytest.mark.gpu

TOL = 1e-12  # a few steps: the bar of the single operators
LENGTHS = (16, 32, 48, 64, 80, 96, 128)


def field(p, complex_):
    """O(1) on every face, so the face copies of phi count."""
    x, y, z = dbecpy.grid(p)
    X, Y, Z = np.meshgrid(x, y, z, indexing="ij")
    f = 1.0 + 0.4 * np.cos(0.7 * X + 0.3 * Y) * np.sin(0.5 * Z + 0.2) + 0.1 * X / (1 + Y * Y)
    return f * np.exp(1j * (0.3 * X - 0.2 * Z)) if complex_ else f


def check(hip_lib, oracle_lib, n):
    p = params(n=n, h=tuple(8.0 / k for k in n), dt=0.002, cutoff=3.0)
    for mode in (dbecpy.IMAG, dbecpy.REAL):
        f = field(p, mode == dbecpy.REAL)
        f /= np.sqrt(np.sum(np.abs(f) ** 2) * p.dx * p.dy * p.dz)
        with dbecpy.Solver(hip_lib, p, mode) as g, dbecpy.Solver(oracle_lib, p, mode) as o, \
                dbecpy.Solver(hip_lib, p, mode, dbecpy.MIXED) as m:
            for s in (g, o, m):
                s.set_psi(f)
                s.set_coupling(60.0, 200.0)
                s.calcpsidd2()
            assert rel(g.get_psidd2(), o.get_psidd2()) < TOL, (n, mode)
            assert rel(m.get_psidd2(), o.get_psidd2()) < 1e-5, (n, mode)
            a, b, c = g.step(3), o.step(3), m.step(3)
            if mode == dbecpy.IMAG:
                assert a == pytest.approx(b, rel=TOL)
                assert c == pytest.approx(b, rel=1e-5)
            assert rel(g.get_psi(), o.get_psi()) < TOL, (n, mode)
            assert rel(m.get_psi(), o.get_psi()) < 1e-5, (n, mode)


@pytest.mark.parametrize("ny", LENGTHS)
def test_every_plane(hip_lib, oracle_lib, ny):
    print(f"[gpu-case] planes {ny} x {LENGTHS}", flush=True)
    for nz in LENGTHS:
        check(hip_lib, oracle_lib, (48 if ny * nz > 96 * 96 else 16, ny, nz))


@pytest.mark.parametrize("n", [(128, 32, 32), (256, 16, 32), (320, 32, 16), (192, 48, 64), (96, 128, 16)],
                         ids=lambda n: "x".join(map(str, n)))
def test_plane_counts(hip_lib, oracle_lib, n):
    print(f"[gpu-case] plane count, grid {n}", flush=True)
    check(hip_lib, oracle_lib, n)

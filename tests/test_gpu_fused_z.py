"""The z sweep fused with the next step's forward z transform, for every z
length: three steps in one call (which run it twice) against three calls (which
run the sweep and the transform as kernels of their own) and against the
oracle.  160 rows of y leave the last workgroup of a plane a part of its rows
where it takes 64 of them, and are too many for the kernels that hold a plane
in LDS."""
import numpy as np
import pytest

import dbecpy
from conftest import params, rel
from test_gpu_plane import field

pytestmark = pytest.mark.gpu

# a few steps: FP64 the bar of the single operators; FP32 a few roundings per
# transform and sweep, the bar of the mixed form
TOL = {dbecpy.FP64: 1e-12, dbecpy.MIXED: 1e-5}


@pytest.mark.parametrize("nz", (16, 32, 48, 64, 80, 96, 128, 160, 192, 256, 320, 384, 512))
def test_every_length(hip_lib, oracle_lib, nz):
    print(f"[gpu-case] fused z, 16 x 160 x {nz}", flush=True)
    n = (16, 160, nz)
    p = params(n=n, h=tuple(8.0 / k for k in n), dt=0.002, cutoff=3.0)
    for mode in (dbecpy.IMAG, dbecpy.REAL):
        f = field(p, mode == dbecpy.REAL)
        f /= np.sqrt(np.sum(np.abs(f) ** 2) * p.dx * p.dy * p.dz)

        def run(lib, prec, calls):
            with dbecpy.Solver(lib, p, mode, prec) as s:
                s.set_psi(f)
                s.set_coupling(60.0, 200.0)
                for k in calls:
                    s.step(k)
                return s.get_psi()

        want = run(oracle_lib, dbecpy.FP64, (3,))
        for prec in (dbecpy.FP64, dbecpy.MIXED):
            a, b = run(hip_lib, prec, (3,)), run(hip_lib, prec, (1, 1, 1))
            assert rel(a, want) < TOL[prec], (nz, mode, prec)
            assert rel(a, b) < TOL[prec], (nz, mode, prec)


def test_from_the_largest_x(hip_lib):
    """Complex psi of 176 MiB or more is swept from the largest x down."""
    n = (96, 512, 256)
    print(f"[gpu-case] fused z, reversed, {n}", flush=True)
    p = params(n=n, h=tuple(8.0 / k for k in n), dt=0.002, cutoff=3.0)
    f = field(p, True)
    f /= np.sqrt(np.sum(np.abs(f) ** 2) * p.dx * p.dy * p.dz)
    assert f.nbytes >= 176 << 20
    out = []
    for calls in ((3,), (1, 1, 1)):
        with dbecpy.Solver(hip_lib, p, dbecpy.REAL, dbecpy.FP64) as s:
            s.set_psi(f)
            s.set_coupling(60.0, 200.0)
            for k in calls:
                s.step(k)
            out.append(s.get_psi())
    assert rel(out[0], out[1]) < TOL[dbecpy.FP64]

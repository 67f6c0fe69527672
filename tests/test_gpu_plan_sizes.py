"""Lengths whose x convolution or fused inverse z pass takes one radix plan on
small grids and another on large ones: a step on either side of the line
against the oracle, real and complex psi."""
import numpy as np
import pytest

import dbecpy
from conftest import params, rel
from test_gpu_fused_z import TOL
from test_gpu_plane import field

pytestmark = pytest.mark.gpu

# x convolution: Ny (Nz/2 + 1) lines, 320 at 4096 (FP64) and 8192 (FP32), 512 at
# 4096 (FP32); inverse z: Nx Ny rows, 320 at 4096 and 12288, complex 160 at 8192 (FP64)
GRIDS = [(320, 16, 160), (320, 64, 160), (320, 128, 160), (512, 16, 160), (512, 48, 192),
         (16, 160, 160), (64, 160, 160), (16, 160, 320), (32, 160, 320), (80, 160, 320)]


@pytest.mark.parametrize("n", GRIDS, ids=lambda n: "x".join(map(str, n)))
def test_either_side(hip_lib, oracle_lib, n):
    print(f"[gpu-case] radix plans by grid size, {n}", flush=True)
    p = params(n=n, h=tuple(8.0 / k for k in n), dt=0.002, cutoff=3.0)
    for mode in (dbecpy.IMAG, dbecpy.REAL):
        f = field(p, mode == dbecpy.REAL)
        f /= np.sqrt(np.sum(np.abs(f) ** 2) * p.dx * p.dy * p.dz)

        def run(lib, prec):
            with dbecpy.Solver(lib, p, mode, prec) as s:
                s.set_psi(f)
                s.set_coupling(60.0, 200.0)
                s.step(1)
                return s.get_psi()

        want = run(oracle_lib, dbecpy.FP64)
        for prec in (dbecpy.FP64, dbecpy.MIXED):
            assert rel(run(hip_lib, prec), want) < TOL[prec], (n, mode, prec)

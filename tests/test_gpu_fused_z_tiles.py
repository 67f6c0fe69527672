"""The z sweep fused with the next step's forward z transform, complex rows, in
launches of several rounds of the chip, where they pass through half tiles (the
launches of test_gpu_fused_z.py take whole ones): three steps in one call
against three calls, which run the sweep and the transform as kernels of their
own.  Rows per length: past the count from which both precisions, or FP64
alone below 256, take half tiles."""
import numpy as np
import pytest

import dbecpy
from conftest import params, rel
from test_gpu_fused_z import TOL
from test_gpu_plane import field

pytestmark = pytest.mark.gpu

ROWS = {16: (320, 512), 32: (256, 320), 48: (256, 160), 64: (256, 320), 80: (128, 160), 96: (128, 160), 128: (96, 160),
        160: (64, 160), 192: (64, 160), 256: (80, 160), 320: (80, 160), 384: (80, 160), 512: (48, 160)}


@pytest.mark.parametrize("nz", sorted(ROWS))
def test_half_tiles(hip_lib, nz):
    n = (*ROWS[nz], nz)
    print(f"[gpu-case] fused z, half tiles, {n}", flush=True)
    p = params(n=n, h=tuple(8.0 / k for k in n), dt=0.002, cutoff=3.0)
    f = field(p, True)
    f /= np.sqrt(np.sum(np.abs(f) ** 2) * p.dx * p.dy * p.dz)
    for prec in (dbecpy.FP64, dbecpy.MIXED):
        out = []
        for calls in ((3,), (1, 1, 1)):
            with dbecpy.Solver(hip_lib, p, dbecpy.REAL, prec) as s:
                s.set_psi(f)
                s.set_coupling(60.0, 200.0)
                for k in calls:
                    s.step(k)
                out.append(s.get_psi())
        assert rel(out[0], out[1]) < TOL[prec], (n, prec)

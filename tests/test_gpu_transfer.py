"""Fields between host arrays and the device (set_psi, get_psi, get_psidd2, the
3-D density): the plain way and the staged one, at sizes around a staging
piece, in both precisions, and from several threads on several contexts."""
import threading

import numpy as np
import pytest

import dbecpy
from conftest import params

pytestmark = pytest.mark.gpu

# device bytes of psi from 64 KiB (plain) over 1-4 MiB (the plain limits) to 78 MiB;
# 160x96x80 and 320x96x80 leave a last piece shorter than the others
GRIDS = [(16, 32, 16), (64, 64, 32), (64, 64, 64), (80, 96, 80), (160, 96, 80), (320, 96, 80), (256, 160, 128)]


def noise(n, mode, seed):
    r = np.random.default_rng(seed)
    f = r.standard_normal(n)
    return f + 1j * r.standard_normal(n) if mode == dbecpy.REAL else f


def stored(f, prec):
    if prec == dbecpy.FP64:
        return f
    return f.astype(np.complex64 if np.iscomplexobj(f) else np.float32).astype(f.dtype)


def round_trip(lib, n, mode, prec, seed):
    p = params(n=n, h=(0.2, 0.2, 0.2), cutoff=4.0)
    with dbecpy.Solver(lib, p, mode, prec) as s:
        for k in range(2):
            f = noise(n, mode, seed + k)
            s.set_psi(f)
            g = stored(f, prec)
            assert np.array_equal(s.get_psi(), g)
            d = s.density(dbecpy.DEN_XYZ).reshape(n)
            assert np.allclose(d, np.abs(g) ** 2, rtol=1e-15, atol=0)
            s.calcpsidd2()
            a = s.get_psidd2()
            assert a.shape == tuple(n) and np.array_equal(a, s.get_psidd2())


@pytest.mark.parametrize("n", GRIDS, ids=lambda n: "x".join(map(str, n)))
def test_round_trip(hip_lib, n):
    for mode in (dbecpy.IMAG, dbecpy.REAL):
        for prec in (dbecpy.FP64, dbecpy.MIXED):
            print(f"[gpu-case] transfer {n} mode {mode} prec {prec}", flush=True)
            round_trip(hip_lib, n, mode, prec, 11)


def test_threads(hip_lib):
    """More calls at once than the staging pool has slots for."""
    print("[gpu-case] transfers from 4 threads", flush=True)
    bad = []

    def work(k):
        try:
            for _ in range(3):
                round_trip(hip_lib, (128, 128, 96), dbecpy.REAL if k % 2 else dbecpy.IMAG,
                           dbecpy.MIXED if k // 2 else dbecpy.FP64, 100 * k)
        except Exception as e:  # reported by the test's thread
            bad.append(repr(e))

    th = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad

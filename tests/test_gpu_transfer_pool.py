"""Transfers past 32 MiB of host values, which the staging pool's threads share
with the caller, from several host threads at once: contexts come and go, so
the pool stops and starts under them.  The plain limits are 6 MiB (fetch) and
32 MiB (store) of device bytes in FP64, 1.5 and 4 MiB in FP32."""
import threading

import pytest

import dbecpy
from test_gpu_transfer import round_trip

pytestmark = pytest.mark.gpu

GRID = (256, 160, 128)  # 40 MiB of host values, 80 MiB complex


def test_pool_is_shared(hip_lib):
    print("[gpu-case] transfers past 32 MiB from 3 threads", flush=True)
    bad = []

    def work(k):
        try:
            for i in range(2):
                round_trip(hip_lib, GRID, dbecpy.REAL if (k + i) % 2 else dbecpy.IMAG,
                           dbecpy.MIXED if k == 1 else dbecpy.FP64, 10 * k + i)
        except Exception as e:  # reported by the test's thread
            bad.append(repr(e))

    th = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad


def test_last_context_ends_right_after_its_transfer(hip_lib):
    for k in range(3):
        print(f"[gpu-case] transfer, then the end of the only context, {k}", flush=True)
        round_trip(hip_lib, GRID, dbecpy.IMAG, dbecpy.FP64, 50 + k)

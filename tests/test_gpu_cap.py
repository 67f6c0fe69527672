"""A request's status against the growth cap of the mixed ground state: the cap
is flagged where a stored value meets it, not where the faces' own potential
would, which the periodic face copies replace.  16^3 in a flat box, with a
dipolar coupling that makes the second step's exponent peak there: at gd = -1000
it is 42 at most on the stored values and 88 with the faces' own potential (a
restatement in FP64), so the cap of 80 is not met; at -1400 it is 153."""
import pytest

import dbecpy
import dbecserve as ds

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gd,status", [(-1000.0, ds.NOT_CONVERGED), (-1400.0, ds.DIVERGED)])
def test_capped_where_stored(hip_lib, gd, status):
    print(f"[gpu-case] growth cap, gd {gd}", flush=True)
    r = ds.make_request(0, 16, dbecpy.IMAG, dbecpy.MIXED, 0.0, 0.0, (2.4, 2.4, 1.9), 0.007, 2, cutoff=0.14)
    r.dx, r.dy, r.dz, r.gd = 0.06, 0.55, 0.18, gd
    with ds.Server(hip_lib, max_batch=1, check_every=2) as srv:
        got = srv.run_all([r], timeout=60)
    assert got[0]["steps"] == 2
    assert got[0]["status"] == status

"""Host paths of the library that need no device: transfers through the staging
slots and the pool of threads, and which kernels a step launches.
host_paths.cpp stands in for the HIP runtime (its entry points come before the
real ones in symbol lookup) and runs one scenario a process."""
import os
import subprocess

import pytest

import dbecpy
from conftest import PKG, REPO


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not os.path.exists(dbecpy.HIP_LIB):
        pytest.fail(f"{dbecpy.HIP_LIB} is not built; run __graft_entry__.build()")
    exe = str(tmp_path_factory.mktemp("host_paths") / "host_paths")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(REPO, "include"), "-rdynamic", "-o", exe,
                    os.path.join(REPO, "tests", "host_paths.cpp"), "-L" + PKG, "-ldbec_hip", "-Wl,-rpath," + PKG,
                    "-pthread", "-ldl"], check=True)
    return exe


def run(program, scenario, *args, **env):
    keep = {k: v for k, v in os.environ.items() if not k.startswith("DBEC_")}
    r = subprocess.run([program, scenario, *args], env={**keep, "DBEC_AUTOTUNE": "0", **env}, capture_output=True, text=True,
                       timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr[-1000:])


def test_last_context_ends_before_the_pool_has_started(program):
    """The caller may finish a transfer before a thread it started has run; the
    end of the last context then still has to end that thread."""
    run(program, "late_threads")


def test_no_memory_during_a_fetch(program):
    """Slots go back to the pool only when no copy into them is pending, also
    where every allocation after the first copy fails."""
    run(program, "memory")


def test_contexts_of_several_threads(program):
    """Four threads whose transfers, past the bound from which the pool's
    threads help, run at once, while contexts come and go under them."""
    run(program, "callers")


def test_slots_move_between_devices(program):
    """Contexts on five devices, one transfer at a time, with slots for two
    devices' transfers in the pool: none is left to the plain way."""
    run(program, "devices")


def test_noalloc_density_allocates_nothing(program):
    """dbec_density_noalloc up to its largest extract: no device or host memory
    and no event."""
    run(program, "noalloc")


def test_output_steps_up_to_the_largest(program):
    run(program, "long_steps")


def test_fuse_z_switch(program):
    """DBEC_FUSE_Z=0 runs a step's z sweep and the next one's forward z pass as
    two kernels, on the grids of the plane kernels too."""
    run(program, "fused")
    run(program, "unfused", DBEC_FUSE_Z="0")


@pytest.mark.parametrize("prec,tile_kb", [(dbecpy.FP64, 33), (dbecpy.MIXED, 17)], ids=["fp64", "mixed"])
def test_bounds_of_the_z_sweep_rows(program, prec, tile_kb):
    """DBEC_SWEEP_Z_THREADS and DBEC_SWEEP_Z_TILE_KB bound the rows of the fused
    kernel of complex lines as those of real ones: by default 16 rows of 256
    (16 threads each, a tile of 8 rows), 8 below a bound that 16 do not meet,
    and the two kernels where 8 do not meet it either."""
    for want, bound in (("256", {}), ("128", {"DBEC_SWEEP_Z_THREADS": "128"}), ("0", {"DBEC_SWEEP_Z_THREADS": "64"}),
                        ("256", {"DBEC_SWEEP_Z_TILE_KB": str(tile_kb)}),
                        ("128", {"DBEC_SWEEP_Z_TILE_KB": str(tile_kb - 1)}),
                        ("0", {"DBEC_SWEEP_Z_TILE_KB": str(tile_kb // 2 - 1)})):
        run(program, "rows", str(prec), want, **bound)


def test_whole_and_half_tiles(program):
    run(program, "tiles")


def test_small_densities_in_one_slab(program):
    run(program, "one_slab")


def test_tuner_times_the_kernels_that_run(program):
    run(program, "tuned", DBEC_AUTOTUNE="1")

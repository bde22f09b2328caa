"""The tile passes' short arithmetic (csrc/wc_arith.hpp) has the bits of the IEEE operations that the reference's steps use.

* square root and reciprocal, five and three instructions: every float of the range that squared distances, densities and
  distances lie in, on the GPU against sqrtf and 1 / x (and values of all kinds against numpy);
* the pair pressure with its half moved into the mass, on the CPU: equal for every mass the passes run with (magnitudes of
  2^-100 to 2^40), not for masses whose half is not exact.

Positions of these passes are 0 or within [2^-20, 2^20] in magnitude, so squared distances are 0 or within [2^-86, 2^44];
velocities, densities and pressures 0 or within [2^-40, 2^40], as for the shared-reciprocal division of the other passes."""
import ctypes as C
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

HERE = Path(__file__).resolve().parent
LIB = HERE / "libarith_check.so"


@pytest.fixture(scope="module")
def arith():
    if not LIB.exists():
        import __graft_entry__

        __graft_entry__.build_arith_check()
    return C.CDLL(str(LIB))


@pytest.mark.gpu
def test_every_float(arith):
    n, roots, reciprocals = C.c_ulonglong(), C.c_ulonglong(), C.c_ulonglong()
    print("case every float of [2^-96, 2^60)", flush=True)
    assert arith.arith_compare(C.byref(n), C.byref(roots), C.byref(reciprocals)) == 0
    assert n.value == 156 << 23
    assert roots.value == 0 and reciprocals.value == 0


@pytest.mark.gpu
def test_values_against_numpy(arith):
    """What both sides of the comparison above share, the compiler's sqrtf and division, against the host's; and 0 and NaN."""
    rng = np.random.default_rng(5)
    x = np.ldexp(1 + rng.random(1 << 20), rng.integers(-96, 60, 1 << 20)).astype(np.float32)
    edges = np.ldexp(np.float32(1), np.arange(-96, 60)).astype(np.float32)
    x = np.concatenate([x, edges, np.nextafter(edges, np.float32(np.inf)), np.nextafter(edges[1:], np.float32(0))])
    extra = np.array([0.0, np.nan], np.float32)
    v = np.concatenate([x, extra])
    root, rec = np.empty_like(v), np.empty_like(v)
    ptr = lambda a: a.ctypes.data_as(C.c_void_p)
    print(f"case {len(v)} values", flush=True)
    assert arith.arith_values(ptr(v), ptr(root), ptr(rec), len(v)) == 0
    n = len(x)
    assert np.array_equal(root[:n].view(np.uint32), np.sqrt(x).view(np.uint32))
    assert np.array_equal(rec[:n].view(np.uint32), (np.float32(1) / x).view(np.uint32))
    assert root[n].view(np.uint32) == 0 and np.isnan(root[n + 1]) and np.isnan(rec[n + 1])


@pytest.mark.parametrize("lo,hi,equal", [(-100, 40, True), (-100, -98, True), (38, 40, True), (-149, -140, False)])
def test_half_the_mass(tmp_path, lo, hi, equal):
    if shutil.which("gcc") is None:
        pytest.skip("gcc not available")
    exe = tmp_path / "half_mass"
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", str(HERE / "half_mass.c"), "-o", str(exe), "-lm"], check=True)
    r = subprocess.run([str(exe), "2000000", "7", str(lo), str(hi)], capture_output=True, text=True, check=True, timeout=120)
    total, bad = map(int, r.stdout.split())
    assert total == 2_000_000
    assert (bad == 0) == equal, bad

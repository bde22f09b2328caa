"""The library's choices by size and density (csrc/wc_choose.hpp), on the CPU: box shapes of the tile passes, and which
contexts start with them, and the tuner's candidates.  Expected values are the faster of both sides as measured (the header names the times)."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

HERE = Path(__file__).parent
CSRC = HERE.parent / "watercube_amd" / "csrc"


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    exe = tmp_path_factory.mktemp("choose") / "choose"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I", str(CSRC), str(HERE / "choose_main.cpp"), "-o",
                    str(exe)], check=True)
    return exe


@pytest.fixture(scope="module")
def choose(exe):
    def run(*contexts):
        """Each context a list of scenes (n, R, bin, h, rest density, mass); (starts, shape) of each."""
        text = "".join(f"{len(c)} " + " ".join(str(v) for s in c for v in s) + "\n" for c in contexts)
        r = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True)
        rows = [list(map(int, ln.split())) for ln in r.stdout.splitlines()]
        assert len(rows) == len(contexts)
        return [(bool(a), tuple(b)) for a, *b in rows]

    return run


def _block(n, cell, neighbours=None, fill=0.7):
    """A block of n particles with `cell` a cell at rest density; the kernel radius from the neighbours."""
    s = fill / n ** (1 / 3)
    R = max(1, round(1 / (cell ** (1 / 3) * s)))
    h = (neighbours / 4.18879) ** (1 / 3) * s if neighbours else 1 / R
    return n, R, cell ** (1 / 3) * s, h, 1000.0, 1000.0 * s ** 3


STARTS = [
    # ordinary scenes, from the smallest that start so
    (50_000, 8, None, True), (49_999, 8, None, False), (64_000, 8, None, True), (192_000, 12, None, True),
    (1_000_000, 8, None, True), (17_800_000, 8, None, True), (80_000, 20, None, True), (1_500_000, 13, None, True),
    # boxes that do not fit LDS
    (64_000, 38, None, False), (250_000, 46, None, False), (250_000, 104, None, False), (1_000_000, 37, None, False),
    # lists that do not hold the neighbours (512, 256 and 128 entries)
    (1_000_000, 33, 268, False), (4_500_000, 33, 151, False), (9_000_000, 30, 124, False), (250_000, 33, 142, True),
    (4_500_000, 15, 130, False), (700_000, 15, 240, False), (100_000, 10, 480, True), (100_000, 20, 480, False),
    # lanes that idle: 16 to 20, to 22.5, to 28 and more a cell
    (343_000, 17, None, True), (700_000, 17, None, False), (2_000_000, 19, None, False), (1_000_000, 21.4, None, True),
    (2_000_000, 21, None, False), (700_000, 27, None, True), (4_500_000, 26.7, 112, True), (700_000, 30, None, True),
    (1_000_000, 30.5, None, False), (2_000_000, 33, None, False), (4_500_000, 14.8, None, True),
    # ... with a smaller kernel radius
    (1_480_000, 17, 42, True), (3_000_000, 18, 44, False), (1_480_000, 21, 52, True), (3_000_000, 31.5, 78, True),
    (804_000, 31, 101, True),
]


def test_start(choose):
    got = choose(*[[_block(n, cell, nb)] for n, cell, nb, _ in STARTS])
    for (n, cell, nb, want), (starts, _) in zip(STARTS, got):
        ball = min(27.0, 4.18879) * cell  # kernel radius of a cell's side where none is named
        assert starts == want, f"{n} particles, {cell} a cell, {nb or round(ball)} neighbours"


def test_start_of_batches(choose):
    light, dense = _block(100_000, 8), _block(100_000, 46)
    empty = (0,) + light[1:]
    got = choose([light] * 8, [light] * 9 + [dense], [light] * 8 + [dense] * 2, [light, empty], [empty, empty],
                 [_block(19_000, 8)] * 5, [_block(21_000, 8)] * 5, [light] * 45 + [_block(100_000, 20, 300)])
    assert [s for s, _ in got] == [True, True, False, True, False, False, True, False]


def test_densities_that_parameters_do_not_name(choose):
    """Without a usable rest density the grid's mean fill counts, and where it is the larger of the two."""
    n, R = 200_000, 30
    bin_ = 1 / R
    got = choose([(n, R, bin_, bin_, 0.0, 1e-3)], [(n, R, bin_, bin_, 1000.0, 0.0)], [(n, 10, 0.1, 0.1, 0.0, 1e-3)],
                 [(n, 10, 0.1, 0.1, 1.0, 1e-3)], [(n, R, bin_, bin_, -1.0, 1e-3)], [(n, R, bin_, bin_, float("nan"), 1e-3)],
                 # the reference application's own parameters: 0.7 a cell at rest density, 8.6 in the mean
                 [(80_000, 21, 1 / 21, 0.04, 500.0, 0.08)])
    assert [s for s, _ in got] == [True, True, False, False, True, True, True]


def test_box_shapes(choose):
    """Every shape fits LDS at rest density or is the smallest; the lines between them as measured."""
    def shape(n, cell):
        return choose([_block(n, cell)])[0][1]

    assert shape(125_000, 8) == (4, 3, 4) and shape(91_000, 8) == (2, 2, 4)
    assert shape(192_000, 12) == (4, 2, 4) and shape(125_000, 12) == (2, 2, 4)
    assert shape(60_000, 20) == (2, 2, 2) and shape(343_000, 20) == (2, 2, 2) and shape(1_000_000, 19) == (2, 2, 4)
    assert shape(80_000, 15.5) == (2, 2, 4) and shape(1_000_000, 30) == (2, 2, 2)
    cap = {(4, 3, 4): 1920, (4, 2, 4): 1920, (2, 2, 4): 2304}
    for n in (1000, 60_000, 250_000, 1_000_000, 9_000_000):
        for cell in np.geomspace(0.1, 300, 60):
            t = shape(n, cell)
            if t in cap:
                halo = (t[0] + 2) * (t[1] + 2) * (t[2] + 2)
                assert halo * cell <= cap[t], (n, cell, t)
            else:
                assert t == (2, 2, 2)


def test_tuner_candidates(exe):
    """The fastest pair of each mode, and the tile passes (the last variant) together: neither of them in another pair."""
    def candidates(tiles, t):
        text = f"{len(t[0][0])} {int(tiles)} " + " ".join(str(x) for m in t for p in m for x in p)
        r = subprocess.run([str(exe), "tune"], input=text, capture_output=True, text=True, check=True)
        return [tuple(map(int, ln.split())) for ln in r.stdout.splitlines()]

    # [lists][pass][variant], three per-particle variants and the tiles
    t = [[[0.050, 0.048, 0.052, 0.040], [0.060, 0.066, 0.063, 0.070]], [[0.055, 0.057, 0.054, 0.041], [0.041, 0.044, 0.040, 0.029]]]
    assert candidates(True, t) == [(1, 0, 0), (2, 2, 1), (3, 3, 1)]
    assert candidates(False, t) == [(1, 0, 0), (2, 2, 1)]
    # too far behind the least sum (0.070): more than 1.3 of it and 0.05 ms
    t = [[[0.09, 0.04, 0.05, 0.04], [0.06, 0.06, 0.07, 0.03]], [[0.1, 0.1, 0.1, 0.05], [0.042, 0.07, 0.041, 0.03]]]
    t[1][0] = [0.09, 0.1, 0.1, 0.05]
    assert candidates(True, t) == [(1, 0, 0), (0, 2, 1), (3, 3, 1)]
    t[1][0] = [0.12, 0.13, 0.14, 0.05]
    assert candidates(True, t) == [(1, 0, 0), (3, 3, 1)]
    t[0][1] = [0.3] * 3 + [0.03]
    assert candidates(True, t) == [(3, 3, 1)] and candidates(False, t) == [(0, 2, 1)]


def test_descriptor_of_the_tile_variant():
    """The last variant has no workgroup, list length and slots in flight of its own: none are reported."""
    from watercube_amd import _lib as L

    v = L.variants()
    assert v[-1] == (0, 0, 0, 0) and all(b in (64, 128, 256) and c > 0 and k > 0 for b, c, k, _ in v[:-1])

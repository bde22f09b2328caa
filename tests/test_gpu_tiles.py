"""The tile passes (the last tuning variant) against the oracle, bit for bit, at the edges of their boxes."""
import ctypes as C

import numpy as np
import pytest

from watercube_amd import Fluid
from watercube_amd import _lib as L
from watercube_amd.scenes import scaled_block
from watercube_amd.scenes import workload

pytestmark = pytest.mark.gpu



def _clustered(oracle_params, parts, cells, seed):
    """`parts` and clusters of m particles inside the grid cells `cells` = [(cell, m)], shuffled."""
    rng = np.random.default_rng(seed)
    b = float(oracle_params.bin_size)
    add = []
    for cell, m in cells:
        rec = np.zeros(m, L.PARTICLE_DTYPE)
        lo = np.array(cell, np.float64) * b
        rec["position"] = rng.uniform(lo + 0.05 * b, lo + 0.95 * b, (m, 3)).astype(np.float32)
        add.append(rec)
    out = np.concatenate([parts] + add)
    return out[rng.permutation(len(out))]


def _case(name):
    if name == "2x2x4, 12 a cell":  # sides that no box divides
        return scaled_block((23, 17, 19), 0.027, 1, 2.3)
    if name == "2x2x2, 51 a cell":  # more neighbours than the context's lists hold
        return scaled_block((23, 17, 19), 0.027, 1, 3.5)
    if name == "4x2x4, 12 a cell":
        return scaled_block((75, 73, 75), 0.01, 2, 2.3)
    if name == "4x3x4":
        return scaled_block((53, 57, 59), 0.0151, 3)
    if name == "one cell":  # a grid that is a single box
        p, parts = scaled_block((4, 5, 4), 0.2, 4)
        p.grid_res = 1
        p.bin_size = p.size
        return p, parts
    small = name.startswith("small")
    p, parts = scaled_block((20, 20, 20) if small else (53, 57, 59), 0.03 if small else 0.0151, 5)
    if "split" in name:    # boxes over the records that LDS holds: parts of 2x2x2, single cells
        cells = [((3, 3, 2), 900), ((6, 4, 4), 700), ((7, 7, 7), 500)]
    elif "long" in name:   # lists at and over their 512 entries, a cell that fits LDS
        cells = [((5, 5, 5), 513), ((2, 9, 3), 514), ((9, 2, 9), 800)]
    else:                  # a cell over them, searched directly; its neighbours too
        cells = [((5, 5, 5), 2600), ((8, 2, 3), 2305)]
    parts = _clustered(p, parts, cells, 7)
    if "odd positions" in name:  # a box with a position outside the shared arithmetic's range, NaN among them
        parts["position"][11] = (1e-12, 0.2, 0.2)
        parts["position"][12] = (np.nan, 0.1, 0.1)
        parts["position"][13] = (5.0, -3.0, 0.4)
    p.num_particles = len(parts)
    return p, parts


CASES = ["2x2x4, 12 a cell", "2x2x2, 51 a cell", "4x2x4, 12 a cell", "4x3x4", "one cell", "small, split", "small, long", "small, direct",
         "small, split, odd positions", "4x3x4, split", "4x3x4, direct"]


@pytest.mark.parametrize("case", CASES)
def test_tile_passes_bit_exact(case, oracle):
    """Two steps by the tile passes, then one with their density pass writing the context's lists for the
    per-particle force pass: the oracle's bits (NaN where it has NaN), and its cells."""
    p, parts = _case(case)
    print(f"case {case}: n={p.num_particles} R={p.grid_res}", flush=True)
    dt = 2e-6
    st = oracle.OracleState(p, parts)
    tile = L.lib().wc_num_variants() - 1
    with Fluid(p, parts) as f:
        for steps, tuning in ((1, (tile, tile, 0)), (1, (tile, tile, 1)), (1, (tile, 2, 1))):
            f.set_tuning(*tuning)
            st.step(dt, steps)
            f.step(dt, steps)
            f.synchronize()
            got = f.particles(1)
            for k in ("density", "pressure", "velocity", "position"):
                x, y = got[k], st.buf1[k]
                assert np.array_equal(np.isnan(x), np.isnan(y)), f"{case} {tuning}: {k} NaN"
                bad = (x.view(np.uint32) != y.view(np.uint32)) & ~np.isnan(y)
                assert not bad.any(), f"{case} {tuning}: {k} differs at {int(bad.sum())} places"
            assert np.array_equal(f.sort_.getCountBuffer(), st.counts)
            assert np.array_equal(f.sort_.getOffsetBuffer(), st.offsets)
        # the lists that the two kinds of density pass write agree
        counts = []
        for variant in (tile, 2):
            f.set_tuning(variant, 2, 1)
            f.sort_.run()
            f.runDensityProg()
            counts.append(f.neighbour_counts())
        assert np.array_equal(counts[0], counts[1])
        if case == "2x2x2, 51 a cell":
            assert (counts[0] == 0xFFFFFFFF).any()


def test_tile_passes_of_several_scenes_with_thin_boxes(oracle):
    """Scenes whose particles fill the cube thinly (their boxes are searched per particle, in chunks of a scene's
    own), one of a single particle and a dense one, advanced together: every scene has the oracle's bits."""
    import ctypes as C

    from watercube_amd.batch import SceneBatch

    scenes = []
    for k, (n, dense) in enumerate(((700, False), (1, False), (0, True), (3000, False), (257, False))):
        p, parts = scaled_block((20, 20, 20), 0.03, 5)
        if not dense:
            rng = np.random.default_rng(k)
            parts = np.zeros(n, L.PARTICLE_DTYPE)
            parts["position"] = rng.uniform(0.01, 0.99, (n, 3)).astype(np.float32)
            p.num_particles = n
        scenes.append((p, parts, 1e-4, "test"))
    print("case batch of", [len(s[1]) for s in scenes], flush=True)
    tile = L.lib().wc_num_variants() - 1
    with SceneBatch(scenes) as b:
        t = L.wc_tuning(tile, tile, 0)
        L.check(L.lib().wc_set_tuning(b.ctx, C.byref(t)), "wc_set_tuning")
        b.step(3)
        b.synchronize()
        for s, (p, parts, dt, _) in enumerate(scenes):
            st = oracle.OracleState(p, parts)
            st.step(dt, 3)
            got = b.scene_particles(s)
            for k in ("density", "pressure", "velocity", "position"):
                assert np.array_equal(got[k].view(np.uint32), st.buf1[k].view(np.uint32)), f"scene {s}: {k}"


def test_latency_of_an_empty_scene_is_zero(oracle):
    """The passes' leading work items are padded to a multiple of the XCD count.  Padding belongs to no scene: a scene
    without particles, the first one here, keeps a latency of 0."""
    from watercube_amd.batch import SceneBatch

    scenes = []
    for k, n in enumerate((0, 700, 257)):
        p, _ = scaled_block((20, 20, 20), 0.03, 5)
        parts = np.zeros(n, L.PARTICLE_DTYPE)
        parts["position"] = np.random.default_rng(k).uniform(0.01, 0.99, (n, 3)).astype(np.float32)
        p.num_particles = n
        scenes.append((p, parts, 1e-4, "test"))
    tile = L.lib().wc_num_variants() - 1
    for variant in (2, tile):
        print(f"case empty scene, variant {variant}", flush=True)
        with SceneBatch(scenes) as b:
            t = L.wc_tuning(variant, variant, 0)
            L.check(L.lib().wc_set_tuning(b.ctx, C.byref(t)), "wc_set_tuning")
            b.step(3)
            b.synchronize()
            lat = b.latency_ms()
        assert lat[0] == 0.0 and (np.asarray(lat[1:]) > 0.0).all(), f"variant {variant}: {lat}"


def test_cube_size_unrelated_to_the_grid(oracle):
    """wc_create takes `size` and `bin_size` as they are.  On a grid a thousand times wider than `size` every neighbour is
    kept: candidates are marked with a margin that has to cover the rounding of coordinates up to the grid's width.
    A neighbour lost at the cutoff hardly shows in the sums, so the lists' lengths are compared too, with those of the
    per-particle pass."""
    n = 40_000
    p, _ = scaled_block((40, 40, 40), 0.02, 6)
    h = 1.0 / 16
    p.num_particles, p.grid_res, p.size, p.bin_size, p.kernel_radius, p.particle_mass = n, 16, 1e-3, h, h, 1000.0 / n
    p.poly6_const, p.spiky_const, p.visc_const = 315 / (64 * np.pi * h ** 9), -45 / (np.pi * h ** 6), 45 / (np.pi * h ** 6)
    parts = np.zeros(n, L.PARTICLE_DTYPE)
    parts["position"] = np.random.default_rng(11).uniform(0.01, 0.99, (n, 3)).astype(np.float32)
    tile = L.lib().wc_num_variants() - 1
    st = oracle.OracleState(p, parts)
    st.step(2e-6, 1)
    counts = []
    for v in (tile, 2):
        print(f"case wide grid, variant {v}", flush=True)
        with Fluid(p, parts) as f:
            f.set_tuning(v, v, 1)
            f.sort_.run()
            f.runDensityProg()
            counts.append(f.neighbour_counts())
            f.runUpdateProg(2e-6)
            f.synchronize()
            got = f.particles(1)
        for k in ("density", "pressure", "velocity", "position"):
            bad = got[k].view(np.uint32) != st.buf1[k].view(np.uint32)
            assert not bad.any(), f"variant {v}: {k} differs at {int(bad.sum())} places"
    assert np.array_equal(counts[0], counts[1]), f"{int((counts[0] != counts[1]).sum())} lists differ"


def test_mass_whose_half_is_not_exact(oracle):
    """The force pass by tiles moves a half from the pair pressure into the mass, which is exact for normal floats
    only.  A mass of three units of the smallest float, with kernel constants that bring densities into the shared
    arithmetic's range: the oracle's bits."""
    p, parts = scaled_block((20, 20, 20), 0.015, 5)
    parts["position"] *= np.float32(100.0)
    parts["velocity"] = np.random.default_rng(4).normal(0, 0.1, parts["velocity"].shape).astype(np.float32)
    p.size, p.kernel_radius = 100.0, 3.0
    L.derive(p)
    p.particle_mass = 3 * 2.0 ** -149
    p.poly6_const, p.spiky_const, p.visc_const = 1e34, -1e37, 1e36
    p.rest_density, p.stiffness = 1e-8, 1.0
    tile = L.lib().wc_num_variants() - 1
    st = oracle.OracleState(p, parts)
    st.step(2e-6, 1)
    assert 2.0 ** -40 < st.buf1["density"].min() and st.buf1["density"].max() < 1.0  # in the range
    print("case subnormal mass", flush=True)
    with Fluid(p, parts) as f:
        for v in (2, tile):
            f.upload(parts)
            f.set_tuning(v, v, 0)
            f.step(2e-6, 1)
            f.synchronize()
            got = f.particles(1)
            for k in ("density", "pressure", "velocity", "position"):
                bad = got[k].view(np.uint32) != st.buf1[k].view(np.uint32)
                assert not bad.any(), f"variant {v}: {k} differs at {int(bad.sum())} places"


@pytest.mark.parametrize("sequence", ["step", "step, lists off, step", "step, sort", "step, other passes",
                                      "profiled", "learned run"])
def test_neighbour_counts_are_those_of_the_last_listing_pass(sequence):
    """wc_get_neighbour_counts answers for the last density pass that ran in list mode, whatever ran after it: by tiles,
    whose steps leave the lists out until they are asked for, as by the per-particle passes."""
    p, parts, dt, _ = workload("dam_break_16k")
    tile = L.lib().wc_num_variants() - 1
    steps = 20 + len(sequence)  # freed memory holds no other sequence's counts
    out = []
    for v in (tile, 2):
        print(f"case {sequence}, variant {v}", flush=True)
        with Fluid(p, parts) as f:
            f.set_tuning(v, v, 1)
            if sequence == "profiled":
                f.profile(dt, steps)
            elif sequence == "learned run":
                st = L.wc_closure_stats()
                L.check(L.lib().wc_closure_run(f.ctx, None, C.c_float(dt), 4, steps, C.c_float(1e30), C.byref(st)), "run")
            else:
                f.step(dt, steps)
            if sequence == "step, lists off, step":
                f.set_tuning(v, v, 0)
                f.step(dt, steps)
            elif sequence == "step, sort":
                f.sort_.run()
            elif sequence == "step, other passes":
                f.set_tuning(2, 2, 0)
                f.sort_.run()
                f.runDensityProg()
            out.append(f.neighbour_counts())
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("n_side,spacing,ratio,tiles", [((40, 40, 40), 0.0175, 2.0, True), ((40, 40, 40), 0.0175, 3.5, False),
                                                       ((40, 40, 40), 0.0175, 4.7, False), ((36, 36, 36), 0.0175, 2.0, False),
                                                       ((100, 100, 100), 0.008, 3.3, False)])
def test_contexts_start_with_the_faster_passes(n_side, spacing, ratio, tiles):
    """The start follows size and density (test_choose.py has the rule's edges): with 46 and 104 particles a cell, or 151
    neighbours at a million, the per-particle passes are up to seven times faster."""
    p, parts = scaled_block(n_side, spacing, 1, ratio)
    with Fluid(p, parts) as f:
        start = f.get_tuning()
    v = L.lib().wc_num_variants() - 1 if tiles else 2
    assert start == (v, v, 0)


@pytest.mark.parametrize("per", [2, 8])
def test_tuner_leaves_the_state_and_its_lists(per, oracle):
    """wc_tune times steps, and restores buffer 1; buffer 2, the cells and the neighbour lists are those of that state
    whichever passes it picks, and the next steps give the oracle's bits."""
    p, parts = scaled_block((30, 30, 30), 0.025, 4)
    n = len(parts)
    p.grid_res = round((n / per) ** (1 / 3))
    p.kernel_radius = 0.999 / p.grid_res
    L.derive(p)
    parts["position"] = np.random.default_rng(2).uniform(0.01, 0.99, (n, 3)).astype(np.float32)
    print(f"case tuner, {per} a cell", flush=True)
    st = oracle.OracleState(p, parts)
    with Fluid(p, parts) as f:
        f.set_tuning(2, 2, 1)
        f.sort_.run()
        f.runDensityProg()
        want = f.particles(2).tobytes(), f.neighbour_counts().tobytes(), f.sort_.getOffsetBuffer().tobytes()
        f.tune(1e-4, reps=2)
        assert f.particles(1).tobytes() == parts.tobytes()
        assert (f.particles(2).tobytes(), f.neighbour_counts().tobytes(), f.sort_.getOffsetBuffer().tobytes()) == want
        f.runUpdateProg(1e-4)
        st.step(1e-4, 1)
        assert np.array_equal(f.particles(1).view(np.uint32), st.buf1.view(np.uint32))
        f.step(1e-4, 3)
        st.step(1e-4, 3)
        assert np.array_equal(f.particles(1).view(np.uint32), st.buf1.view(np.uint32))


def _held(make, count):
    """Bytes of GPU memory that `count` contexts made by make() hold, per context."""
    def free():  # the HIP runtime the library itself is linked with
        a, b = C.c_size_t(), C.c_size_t()
        assert L.lib().hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    before = free()
    made = [make() for _ in range(count)]
    held = before - free()
    for f in made:
        f.close()
    return held / count


@pytest.mark.parametrize("case", ["2,048", "one particle", "16,384", "64,000 per particle", "64,000 tuned off", "2,048 by tiles"])
def test_memory_of_contexts_without_the_tile_passes(case):
    """A context holds the tile passes' buffers (2 KB a particle and more) only if it runs them; few boxes and particles
    need few list chunks."""
    tile = L.lib().wc_num_variants() - 1
    n_side = {"2,048": (16, 16, 8), "one particle": (1, 1, 1), "16,384": (32, 32, 16), "2,048 by tiles": (16, 16, 8)}.get(case, (40, 40, 40))
    p, parts = scaled_block(n_side, 0.015, 1)
    if case == "64,000 tuned off":  # a thin gas, which the tuner finds faster per particle
        p.grid_res, p.kernel_radius = 28, 0.999 / 28
        L.derive(p)
        parts["position"] = np.random.default_rng(1).uniform(0.01, 0.99, (len(parts), 3)).astype(np.float32)

    def make():
        f = Fluid(p, parts).setup()
        if case == "64,000 per particle":
            f.set_tuning(2, 2, 0)
        elif case == "64,000 tuned off":
            f.tune(1e-6, reps=2)
            assert f.get_tuning()[0] != tile
        elif case == "2,048 by tiles":
            f.set_tuning(tile, tile, 0)
        f.step(1e-6, 2)
        f.synchronize()
        return f

    make().close()  # what the library and the runtime load once
    cells = int(p.grid_res) ** 3
    base = 200 * len(parts) + 16 * cells + (260 * len(parts) if case == "64,000 tuned off" else 0)
    # some 24 buffers, a stream and two graphs take 8 MB however small; 2,048 particles 357 list chunks of 64 KB
    limit = base + (12 << 20) + (28 << 20 if case == "2,048 by tiles" else 0)
    held = _held(make, 8)
    print(f"case {case}: {held / 1e6:.1f} MB a context, limit {limit / 1e6:.1f}", flush=True)
    assert held < limit


def test_buffers_follow_the_tuning(oracle):
    """The tile passes' buffers come with the first sort that needs them, also after steps of other passes, a larger grid or
    a tuner's run: the oracle's bits throughout."""
    tile = L.lib().wc_num_variants() - 1
    p, parts = scaled_block((30, 31, 29), 0.02, 3)
    small, _ = scaled_block((30, 31, 29), 0.02, 3, 3.3)  # fewer cells, other boxes
    st = oracle.OracleState(p, parts)
    with Fluid(p, parts) as f:
        def check(what, q=p):
            nonlocal st
            print(f"case {what}", flush=True)
            st = oracle.OracleState(q, st.buf1)
            f.step(2e-5, 2)
            st.step(2e-5, 2)
            f.synchronize()
            assert np.array_equal(f.particles(1).view(np.uint32), st.buf1.view(np.uint32)), what

        check("per particle")
        L.check(L.lib().wc_set_params(f.ctx, C.byref(small)), "wc_set_params")
        f.set_tuning(tile, tile, 1)
        check("tiles, few cells", small)
        L.check(L.lib().wc_set_params(f.ctx, C.byref(p)), "wc_set_params")
        check("tiles, more cells")
        f.set_tuning(2, 2, 1)
        check("per particle again")
        f.tune(1e-7, reps=1)
        check("tuned")
        f.set_tuning(tile, tile, 1)
        f.sort_.run()
        f.runDensityProg()
        f.runUpdateProg(2e-5)
        st.step(2e-5, 1)
        f.synchronize()
        assert np.array_equal(f.particles(1).view(np.uint32), st.buf1.view(np.uint32))
        check("after passes one by one")


def test_kernel_terms_that_overflow(oracle):
    """A pair without positive pressure adds nothing, also when the kernel's term overflows: the force pass by tiles adds 0
    times that term, so contexts with such constants keep the other passes.  The oracle's bits."""
    p, parts = scaled_block((20, 20, 20), 0.015, 5)
    parts["position"] *= np.float32(100.0)
    p.size, p.kernel_radius = 100.0, 3.0
    L.derive(p)
    p.particle_mass, p.rest_density, p.stiffness = 1.0, 1e6, 1.0  # every pressure negative
    p.spiky_const = -3e38  # the nearest neighbours, 1.2 to 1.8 away: (3 - d)^2 times this is infinite
    tile = L.lib().wc_num_variants() - 1
    st = oracle.OracleState(p, parts)
    st.step(1e-3, 2)
    assert np.isfinite(st.buf1["velocity"]).all() and (st.buf1["pressure"] < 0).all()
    print("case kernel term overflows", flush=True)
    with Fluid(p, parts) as f:
        f.set_tuning(tile, tile, 0)
        f.step(1e-3, 2)
        f.synchronize()
        assert np.array_equal(f.particles(1).view(np.uint32), st.buf1.view(np.uint32))


@pytest.mark.parametrize("scene,marks", [("block_1m", (100, 300, 500)), ("block_sphere_17m", (3, 20))])
def test_tile_trajectory_of_the_large_scenes(scene, marks):
    """The benchmark's scenes by the passes that they start on, whose lists hold 256 and 128 entries there, against the
    per-particle passes with lists (which the 500-step comparison with the oracle pins): the same bits all the way."""
    p, parts, dt, _ = workload(scene)
    tile = L.lib().wc_num_variants() - 1
    with Fluid(p, parts) as a, Fluid(p, parts) as b:
        assert a.get_tuning()[:2] == (tile, tile)
        a.set_tuning(tile, tile, 1)
        b.set_tuning(4, 0, 1)
        done = 0
        for upto in marks:
            print(f"case {scene}: steps {done}..{upto}", flush=True)
            a.step(dt, upto - done)
            b.step(dt, upto - done)
            a.synchronize()
            b.synchronize()
            done = upto
            x, y = a.particles(1).view(np.uint32), b.particles(1).view(np.uint32)
            assert np.array_equal(x, y), f"{scene} after {done} steps: {int((x != y).sum())} words differ"


def test_parameters_that_change_the_box_shape(oracle):
    """wc_set_params between steps, with kernel radii whose rest density asks for other boxes each time (and back)."""
    p, parts = scaled_block((40, 37, 41), 0.02, 8)
    tile = L.lib().wc_num_variants() - 1
    st = oracle.OracleState(p, parts)
    with Fluid(p, parts) as f:
        f.set_tuning(tile, tile, 0)
        for ratio in (2.0, 2.7, 2.3, 3.5, 2.0):
            print(f"case kernel radius {ratio}", flush=True)
            q, _ = scaled_block((40, 37, 41), 0.02, 8, ratio)
            L.check(L.lib().wc_set_params(f.ctx, C.byref(q)), "wc_set_params")
            st = oracle.OracleState(q, st.buf1)
            f.step(2e-5, 2)
            st.step(2e-5, 2)
            f.synchronize()
            got = f.particles(1)
            assert np.array_equal(got.view(np.uint32), st.buf1.view(np.uint32)), f"ratio {ratio}"


@pytest.mark.parametrize("n_side", [(40, 40, 40), (20, 20, 20)])
def test_steps_captured_before_the_buffers_go(n_side):
    """A context tuned away from the tile passes gives their buffers back when it next waits; steps captured before that,
    and after, hold no address of them.  The same bits as a context that never had them."""
    p, parts = scaled_block(n_side, 0.0175, 1)
    tile = L.lib().wc_num_variants() - 1
    with Fluid(p, parts) as a, Fluid(p, parts) as b:
        print(f"case buffers given back, {len(parts)} particles", flush=True)
        b.set_tuning(2, 2, 1)
        a.set_tuning(tile, tile, 1)
        a.step(2e-5, 3)
        a.set_tuning(2, 2, 1)
        a.step(2e-5, 9)   # captured with the buffers there
        b.step(2e-5, 12)
        a.synchronize()   # gives them back
        a.step(2e-5, 9)   # replayed or captured again
        a.synchronize()
        a.set_tuning(tile, tile, 0)
        a.step(2e-5, 9)
        b.step(2e-5, 18)
        a.synchronize()
        b.synchronize()
        assert a.particles(1).tobytes() == b.particles(1).tobytes()

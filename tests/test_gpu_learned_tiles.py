"""The learned step by the tile passes (the last tuning variant) against the per-particle passes, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from watercube_amd import Fluid
from watercube_amd import _lib as L
from watercube_amd.closure import ClosureNet, DeviceArray
from watercube_amd.scenes import scaled_block, workload

pytestmark = pytest.mark.gpu


def _tile():
    return L.lib().wc_num_variants() - 1


def _net(scale=0.05):
    net = ClosureNet(max_batch=64)
    net.set_params(np.random.default_rng(21).normal(0, scale, ClosureNet.num_params()).astype(np.float32))
    return net


def _scene(name):
    if name == "dam_break_16k":
        p, parts, dt, _ = workload(name)
        return p, parts, dt
    p, parts = scaled_block((23, 21, 19), 0.01, seed=7, h_over_s=2.0 if name == "ragged" else 3.0)
    return p, parts, 2e-4


SCENES = ["dam_break_16k", "ragged", "dense"]  # dense: lists of more than 64 neighbours


@pytest.mark.parametrize("scene", SCENES)
@pytest.mark.parametrize("lists", [0, 1])
def test_learned_update(scene, lists):
    """wc_closure_update with a correction and the plain acceleration written out."""
    p, parts, dt = _scene(scene)
    n = len(parts)
    corr = np.random.default_rng(1).normal(0, 1, (n, 4)).astype(np.float32)
    cd, acc = DeviceArray((n, 4), np.float32).upload(corr), DeviceArray((n, 4), np.float32)
    out = []
    for v in (2, _tile()):
        print(f"case {scene}, lists {lists}, variant {v}", flush=True)
        with Fluid(p, parts) as f:
            f.track_ids(True)
            f.set_tuning(v, v, lists)
            f.step(dt, 5)
            f.sort_.run()
            f.runDensityProg()
            acc.upload(np.zeros((n, 4), np.float32))
            L.check(L.lib().wc_closure_update(f.ctx, C.c_float(4 * dt), cd.ptr, C.c_float(9.81), acc.ptr), "update")
            f.synchronize()
            out.append((f.particles(1).tobytes(), acc.download()[:, :3].tobytes(), f.ids(1).tobytes()))
    assert out[0] == out[1]
    assert np.frombuffer(out[0][1], np.float32).any()


@pytest.mark.parametrize("scene", SCENES)
@pytest.mark.parametrize("smooth,substeps,tol", [(0, 0, 1e9), (0, 1, 1e9), (1, 0, 1e9), (0, 0, -1.0), (0, 1, 1e-5)],
                         ids=["large", "substeps", "smoothed", "rejected", "judged"])
def test_learned_run(scene, smooth, substeps, tol):
    """wc_closure_run with identities: steps accepted, rejected (restored from what the force pass saved) and both;
    then closure inputs and inference from the lists of the state that it leaves."""
    p, parts, dt = _scene(scene)
    n, K, macro = len(parts), 4, 5
    net = _net()
    out = []
    for v, lists in ((2, 1), (_tile(), 1), (_tile(), 0)):
        print(f"case {scene}, smooth {smooth}, substeps {substeps}, tol {tol}, variant {v}, lists {lists}", flush=True)
        with Fluid(p, parts) as f:
            f.track_ids(True)
            f.set_tuning(v, v, lists)
            L.check(L.lib().wc_closure_set_smoothing(f.ctx, smooth), "smoothing")
            L.check(L.lib().wc_closure_set_integrator(f.ctx, substeps), "integrator")
            st = L.wc_closure_stats()
            L.check(L.lib().wc_closure_run(f.ctx, net.h, C.c_float(dt), K, macro, C.c_float(tol), C.byref(st)), "run")
            if tol < 0:
                assert st.fallbacks == macro
            out.append((f.particles(1).tobytes(), f.particles(2).tobytes(), f.ids(1).tobytes(), st.macro_steps,
                        st.fallbacks, st.max_density_jump, st.peak_density))
    assert out[0] == out[1] and out[0] == out[2]


@pytest.mark.parametrize("scene", SCENES)
def test_inputs_and_inference_after_steps(scene):
    """Steps by tiles leave the neighbour lists out; closure inputs and inference that follow them write them."""
    p, parts, dt = _scene(scene)
    n = len(parts)
    net = _net()
    x, y = DeviceArray((n, 208), np.uint16), DeviceArray((n, 4), np.float32)
    out = []
    for v in (2, _tile()):
        for first in ("features", "infer"):
            print(f"case {scene}, variant {v}, {first} first", flush=True)
            with Fluid(p, parts) as f:
                f.set_tuning(v, v, 1)
                f.step(dt, 9)
                for what in (first, "infer" if first == "features" else "features"):
                    if what == "features":
                        L.check(L.lib().wc_closure_features(f.ctx, C.c_float(4.0), None, 0, x.ptr), what)
                    else:
                        L.check(L.lib().wc_closure_infer(f.ctx, net.h, C.c_float(4.0), y.ptr), what)
                f.step(dt, 3)  # and the steps go on from there
                out.append((x.download().tobytes(), y.download().tobytes(), f.particles(1).tobytes()))
    assert all(o == out[0] for o in out[1:])

"""mh_localize's steps on the device: n steps in one call are n calls of one step,
bit for bit, across the lengths of its chunks; a call's traces are the sums that
mh_point_to_psdf gives at each pose; a frame without a usable point, and a
singular system, end the call as they are met.  Image sizes: four lanes a point
and one, ragged tiles."""
from dataclasses import replace

import numpy as np
import pytest

from meshhashing_amd.configs import C1
from meshhashing_amd.engine import Volume, synth_depth, synth_pose

pytestmark = pytest.mark.gpu


def _volume(w, h):
    cfg = replace(C1, width=w, height=h, fx=0.82 * w, fy=0.82 * w, cx=0.5 * w, cy=0.5 * h)
    vol = Volume(cfg)
    for f in range(3):
        vol.upload_depth(synth_depth(cfg, f), synth_pose(cfg, f))
        vol.alloc()
        vol.collect_visible()
        vol.integrate_tsdf()
    return cfg, vol


@pytest.mark.parametrize("size,steps", [((320, 240), 33), ((97, 75), 5), ((1600, 1200), 3), ((18, 17), 64)])
def test_steps_are_calls_of_one_step(hip_device, size, steps):
    cfg, vol = _volume(*size)
    start = synth_pose(cfg, 1).copy()
    start[:3, 3] += [0.01, -0.008, 0.006]
    vol.upload_depth(synth_depth(cfg, 1), start)
    out = vol.localize(start, iterations=steps, lam=1e3, corrected=True)
    T, err, count = start, [], []
    for _ in range(out["steps"]):
        at = vol.point_to_psdf(T, corrected=True)
        one = vol.localize(T, iterations=1, lam=1e3, corrected=True)
        assert at["err"] == one["err"][0] and at["count"] == one["count"][0]
        err.append(one["err"][0])
        count.append(one["count"][0])
        T = one["wTc"]
    assert out["steps"] == steps and min(count) > 0
    assert np.array_equal(out["wTc"], T)
    assert np.array_equal(out["err"][:steps], err) and np.array_equal(out["count"][:steps], count)


def test_a_call_ends_where_no_step_can_be_taken(hip_device):
    cfg, vol = _volume(320, 240)
    pose = synth_pose(cfg, 1)
    vol.upload_depth(np.zeros((240, 320), np.uint16), pose)
    out = vol.localize(pose, iterations=40, lam=1e3)
    assert out["steps"] == 0 and np.array_equal(out["wTc"], pose.astype(np.float32))
    # the reference's Jacobian has two equal columns: singular without damping
    vol.upload_depth(synth_depth(cfg, 1), pose)
    out = vol.localize(pose, iterations=40, lam=0.0)
    assert out["steps"] == 0 and out["count"][0] > 0 and np.array_equal(out["wTc"], pose.astype(np.float32))
    assert out["err"][0] == vol.point_to_psdf(pose)["err"] and not out["err"][1:].any()
    # and the next call starts afresh
    assert vol.localize(pose, iterations=2, lam=1e3)["steps"] == 2

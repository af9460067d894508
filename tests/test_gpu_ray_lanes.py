"""The raycast's launches of one, two and four lanes a ray: single images against
the oracle's plain march over a ladder of sizes in which neighbours differ by less
than the range of any lane count, so that wherever the lines lie each count is
taken; and batches of one to four scenes, whose scenes share those lines, against
the same scenes run alone (another lane count for the same rays), with meshing
beside the raycast and without it, eager and replayed."""
from dataclasses import replace

import numpy as np
import pytest

from meshhashing_amd.configs import c4_scenes
from meshhashing_amd.engine import Batch, Volume, synth_depth, synth_pose
from test_gpu_batch import assert_same, scene_state
from test_gpu_raycast_views import _compare, _look, room  # noqa: F401

pytestmark = pytest.mark.gpu

# pixels: 76 800 ... 226 000, each at most a third more than the one before
LADDER = [(320, 240), (333, 251), (350, 263), (352, 262), (397, 303), (420, 331), (451, 361), (453, 363), (521, 391),
          (590, 383)]


@pytest.mark.parametrize("size", LADDER)
def test_images_over_the_lane_counts(room, size):  # noqa: F811
    from meshhashing_amd.engine import synth_pose as pose_of
    cfg, vol, orc, g = room
    w, h = size
    p = replace(cfg, width=w, height=h, fx=0.82 * w, fy=0.82 * w, cx=0.5 * w, cy=0.5 * h).raycaster_params()
    rng = np.random.default_rng(w)
    c = (g["pos"][rng.integers(len(g["pos"]))] + 0.5) * 8 * cfg.voxel_size
    off = rng.normal(size=3)
    beside = _look(c + off / np.linalg.norm(off) * 12 * cfg.voxel_size, c)
    hits = [_compare(cfg, vol, orc, T, p)
            for T in (np.linalg.inv(pose_of(cfg, 4).astype(np.float64)).astype(np.float32), beside)]
    assert max(hits) > 0.5


def _images(b, n, px, cast):
    import torch
    d = torch.full((n * px,), -1.0, device="cuda")
    v = torch.full((3 * n * px,), -1.0, device="cuda")
    m = torch.full((3 * n * px,), -1.0, device="cuda")
    cast(d, v, m)
    b.synchronize()
    return [x.cpu().numpy().view(np.uint32).reshape(n, -1) for x in (d, v, m)]


@pytest.mark.parametrize("mesh, graph", [(True, True), (True, False), (False, True)])
@pytest.mark.parametrize("n, w, h", [(1, 320, 240), (2, 320, 240), (1, 397, 303), (4, 161, 119), (3, 97, 71)])
def test_batches_over_the_lane_counts(hip_device, n, w, h, mesh, graph):
    import torch
    cfgs = [replace(c, width=w, height=h, fx=0.82 * w, fy=0.82 * w, cx=0.5 * w, cy=0.5 * h) for c in c4_scenes(n, 3)]
    px, frames = w * h, range(3)
    b = Batch(cfgs)
    out = [torch.empty(n * px, device="cuda"), torch.empty(3 * n * px, device="cuda"), torch.empty(3 * n * px, device="cuda")]
    b.set_raycast(*[x.data_ptr() for x in out])
    got = []
    for f in frames:
        b.frame(np.stack([synth_depth(c, f) for c in cfgs]), np.stack([synth_pose(c, f) for c in cfgs]))
        for x in out:
            x.fill_(-1.0)  # eager work between the replays
        torch.cuda.synchronize()
        b.run(mesh=mesh, raycast=True, graph=graph)
        b.synchronize()
        got.append([x.cpu().numpy().view(np.uint32).reshape(n, -1) for x in out])
    for s, cfg in enumerate(cfgs):
        vol = Volume(cfg)
        for f in frames:
            vol.upload_depth(synth_depth(cfg, f), synth_pose(cfg, f))
            vol.alloc()
            vol.collect_visible()
            vol.integrate_tsdf()
            if mesh:
                vol.marching_cubes()
            one = _images(vol, 1, px, lambda d, v, m: vol.raycast(vol.pose()[1], d.data_ptr(), v.data_ptr(), m.data_ptr()))
            for a, o in zip(got[f], one):
                assert np.array_equal(a[s], o[0]), (s, f)
        assert np.isfinite(one[0].view(np.float32)).mean() > 0.5
        assert_same(scene_state(b.volumes[s], mesh), scene_state(vol, mesh), f"scene {s}")
        vol.close()
    b.close()

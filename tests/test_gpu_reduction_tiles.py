"""The parallel FP64 sums where their launches change: up to 512 rows (one an 8 x 8
tile of the image) go to one workgroup, more to workgroups of 64 rows whose last one
to finish adds up; a last workgroup of one row, of a few, and full ones; and
again on the same volume, for which the count of finished workgroups starts at 0."""
from dataclasses import replace

import numpy as np
import pytest

from meshhashing_amd.configs import C1
from meshhashing_amd.engine import Volume, synth_depth, synth_pose

pytestmark = pytest.mark.gpu

# tiles across x tiles down: 511, 512, 513 (8 x 64 + 1), 576 (9 x 64), 577 rows
TILES = [(73, 7), (32, 16), (27, 19), (24, 24), (577, 1)]


@pytest.mark.parametrize("tiles", TILES)
def test_adjoint_sums(hip_device, tiles):
    import torch
    cfg = replace(C1, frames=20)
    vol = Volume(cfg)
    vol.upload_depth(synth_depth(cfg, 0), synth_pose(cfg, 0))
    vol.alloc()
    vol.collect_visible()
    vol.integrate_tsdf()
    w, h = 8 * tiles[0] - 3, 8 * tiles[1] - 2
    p = replace(cfg, width=w, height=h, cx=0.5 * w, cy=0.5 * h, fx=262.5, fy=262.5).raycaster_params()
    cTw, n = vol.pose()[1], w * h
    d = torch.empty(n, device="cuda")
    vol.raycast(cTw, d.data_ptr(), params=p)
    rng = np.random.default_rng(w)
    for _ in range(2):
        obs = rng.uniform(1.0, 4.0, n).astype(np.float32)
        obs[rng.random(n) < 0.1] = 0.0
        o = torch.from_numpy(obs).cuda()
        # the allocation-free entry point takes images up to 1280 pixels wide
        out = [vol.raycast_backward(cTw, o.data_ptr(), params=p, noalloc=k) for k in (False, w <= 1280)]
        for k in out[0]:
            assert np.array_equal(out[0][k], out[1][k]), k
        dep = d.cpu().numpy()
        use = np.isfinite(dep) & (obs > 0)
        res = (dep[use] - obs[use]).astype(np.float64)
        assert out[0]["observed"] == int((obs > 0).sum())
        assert out[0]["pixels"] == int(use.sum()) > 0
        # two FP64 sums of the same n terms differ by at most n eps of their value
        assert abs(out[0]["loss"] - 0.5 * (res ** 2).sum()) <= n * 2.0 ** -52 * max(out[0]["loss"], 1e-30)


@pytest.mark.parametrize("tiles", TILES)
def test_localiser_sums(hip_device, oracle_mod, tiles):
    w, h = 16 * tiles[0] - 2, 16 * tiles[1] - 2  # a tile has 16 x 16 pixels here
    cfg = replace(C1, frames=20, width=w, height=h, cx=0.5 * w, cy=0.5 * h)
    vol, orc = Volume(cfg), oracle_mod.Oracle(cfg)
    for f in (0, 1):
        vol.upload_depth(synth_depth(cfg, f), synth_pose(cfg, f))
        vol.alloc()
        vol.collect_visible()
        vol.integrate_tsdf()
    g = vol.dump_blocks()
    orc.load_blocks(g["pos"], g["sdf"], g["weight"], g["color"])
    for f in (1, 2):
        start = synth_pose(cfg, f).copy()
        start[:3, 3] += [0.01, -0.008, 0.006]
        vol.upload_depth(synth_depth(cfg, f), start)
        orc.set_frame(synth_depth(cfg, f), start)
        a, r = vol.point_to_psdf(start, corrected=True), orc.point_to_psdf(start, corrected=True)
        assert a["count"] == r["count"] > 0
        for k in ("A", "b", "err"):  # the bar of test_gpu_localize
            assert np.abs(a[k] - r[k]).max() <= 1e-9 * max(np.abs(r[k]).max(), 1e-30), k
        out = vol.localize(start, iterations=2, lam=1e3, corrected=True)
        assert out["steps"] == 2 and out["err"][0] == a["err"] and out["count"][0] == a["count"]

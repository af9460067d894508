"""The raycast from views at which its block ranges, block tables and launch
shapes can go wrong, against the oracle's plain march over the same blocks:
blocks beside, behind and right in front of the camera, images of one tile,
ragged ones and ones larger than the range pass's LDS table, block sets in
linked lists, and a field whose blocks hold both signs, one sign, or nothing."""
from dataclasses import replace

import numpy as np
import pytest

from meshhashing_amd.configs import C1

pytestmark = pytest.mark.gpu


def _compare(cfg, vol, orc, cTw, params):
    import torch
    n = params.width * params.height
    d = torch.empty(n, device="cuda")
    v = torch.empty(3 * n, device="cuda")
    m = torch.empty(3 * n, device="cuda")
    vol.raycast(cTw, d.data_ptr(), v.data_ptr(), m.data_ptr(), params=params)
    vol.synchronize()
    do, vo, no = orc.raycast(cTw, params)
    dg = d.cpu().numpy().reshape(do.shape)
    ng = m.cpu().numpy().reshape(no.shape)
    vg = v.cpu().numpy().reshape(vo.shape)
    hit = np.isfinite(do)
    assert np.array_equal(np.isfinite(dg), hit)
    if hit.any():
        # the bars of test_gpu_parity's raycast
        assert np.abs(dg[hit] - do[hit]).max() <= 1e-4
        assert np.abs(vg[hit] - vo[hit]).max() <= 1e-4
        assert np.abs(ng[hit] - no[hit]).max() < 1e-4
    return hit.mean()


def _look(eye, at):
    f = np.asarray(at, float) - eye
    f /= np.linalg.norm(f)
    r = np.cross(f, [0.0, 1.0, 0.0])
    r /= np.linalg.norm(r)
    T = np.eye(4)
    T[:3, 0], T[:3, 1], T[:3, 2], T[:3, 3] = r, np.cross(f, r), f, eye
    return np.linalg.inv(T).astype(np.float32)


@pytest.fixture(scope="module")
def room(hip_device, oracle_mod):
    from meshhashing_amd.engine import Volume, synth_depth, synth_pose
    cfg = replace(C1, frames=20, bucket_count=450)  # many buckets overflow into lists
    vol = Volume(cfg)
    for f in range(0, 20, 3):
        vol.upload_depth(synth_depth(cfg, f), synth_pose(cfg, f))
        vol.alloc()
        vol.collect_visible()
        vol.integrate_tsdf()
    g = vol.dump_blocks()
    orc = oracle_mod.Oracle(replace(cfg, bucket_count=1 << 14))
    orc.load_blocks(g["pos"], g["sdf"], g["weight"], g["color"])
    return cfg, vol, orc, g


@pytest.mark.parametrize("size", [(8, 8), (61, 47), (320, 240), (331, 253), (705, 521)])
def test_views_of_a_room(room, size):
    from meshhashing_amd.engine import synth_pose
    cfg, vol, orc, g = room
    w, h = size
    view = replace(cfg, width=w, height=h, fx=0.82 * w, fy=0.82 * w, cx=0.5 * w, cy=0.5 * h)
    p = view.raycaster_params()
    rng = np.random.default_rng(w)
    centre = (g["pos"][rng.integers(len(g["pos"]), size=3)] + 0.5) * 8 * cfg.voxel_size
    poses = [np.linalg.inv(synth_pose(cfg, 4).astype(np.float64)).astype(np.float32)]
    for c in centre:  # a block's length from a surface block: beside it, and looking at it
        off = rng.normal(size=3)
        eye = c + off / np.linalg.norm(off) * 8 * cfg.voxel_size * rng.uniform(0.9, 2.5)
        poses += [_look(eye, c), _look(eye, c + rng.normal(size=3))]
    hits = [_compare(cfg, vol, orc, T, p) for T in poses]
    assert max(hits) > 0.5


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_views_of_random_blocks(hip_device, oracle_mod, seed):
    """Scattered blocks (absent neighbours everywhere), fields of both signs,
    positive only, negative only, and with exact zeros."""
    from meshhashing_amd.engine import Volume
    cfg = replace(C1, bucket_count=200, value_capacity=1 << 12, width=96, height=80, fx=90.0, fy=90.0, cx=48.0, cy=40.0)
    rng = np.random.default_rng(seed)
    pos = np.unique(rng.integers(-5, 6, size=(500, 3)), axis=0).astype(np.int32)
    n = len(pos)
    sdf = (rng.normal(size=(n, 512)) * 0.02).astype(np.float32)
    i = np.arange(512)
    lin = (pos[:, 2:3] * 8 + i // 64) * cfg.voxel_size - 0.1
    smooth = rng.random(n) < 0.5
    sdf[smooth] = (-lin[smooth] * 0.3).astype(np.float32)
    kind = rng.integers(0, 6, n)
    sdf[kind == 0] = np.abs(sdf[kind == 0])
    sdf[kind == 1] = -np.abs(sdf[kind == 1])
    sdf[kind == 2] = 0.01
    odd = kind == 3
    sdf[odd] *= (rng.random((odd.sum(), 512)) < 0.9)  # some exact zeros
    weight = np.ones((n, 512), np.float32)
    vol, orc = Volume(cfg), oracle_mod.Oracle(replace(cfg, bucket_count=1 << 12))
    vol.load_blocks(pos, sdf, weight)
    orc.load_blocks(pos, sdf, weight)
    p = cfg.raycaster_params()
    hits = []
    for _ in range(5):
        eye = rng.normal(size=3)
        eye *= rng.uniform(0.6, 2.5) / np.linalg.norm(eye)
        hits.append(_compare(cfg, vol, orc, _look(eye, rng.normal(size=3) * 0.3), p))
    assert max(hits) > 0.02

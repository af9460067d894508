"""Marching cubes over scattered blocks, against the oracle: blocks whose every
cube is crossed (several rounds of slot claims and of the payload queue), blocks
with a few crossings, with one sign, unobserved ones and lone ones, meshed twice
with the field changed in between (slots freed, surfaces lost), and a second
pass over a part of them only (neighbours with stored configurations).  Topology
and vertex positions, bit for bit; normals are left to test_gpu_parity, a noisy
field's gradient being no continuous function of the position."""
from dataclasses import replace

import numpy as np
import pytest

from meshhashing_amd.configs import C1

pytestmark = pytest.mark.gpu


def _fields(rng, n, cfg):
    sdf = np.empty((n, 512), np.float32)
    kind = rng.integers(0, 6, n)
    for i, k in enumerate(kind):
        if k == 0:
            sdf[i] = rng.normal(size=512) * 0.03
        elif k == 1:
            sdf[i] = np.where(np.arange(512) % 2 ^ np.arange(512) // 8 % 2 ^ np.arange(512) // 64 % 2, 0.03, -0.03)
        elif k == 2:
            sdf[i] = (np.arange(512) // 64 - rng.uniform(0, 7)) * cfg.voxel_size
        else:
            sdf[i] = {3: 0.05, 4: -0.05, 5: 0.04}[int(k)]
    weight = np.ones((n, 512), np.float32)
    weight[kind == 5] = 0.0
    return sdf, weight


def _compare(vol, orc):
    assert np.array_equal(vol.dump_cube_indices(), orc.dump_blocks()["cube"])
    g, o = vol.dump_mesh(), orc.dump_mesh()
    for k in ("tri_cube", "tri", "vkey", "vref"):
        assert np.array_equal(g[k], o[k]), k
    assert np.array_equal(g["vval"][:, :3], o["vval"][:, :3].astype(np.float32))
    return len(g["tri"])


@pytest.mark.parametrize("seed, count, spread", [(0, 1, 0), (1, 12, 1), (2, 400, 4), (3, 1500, 6)])
def test_scattered_blocks(hip_device, oracle_mod, seed, count, spread):
    from meshhashing_amd.engine import Volume, synth_depth, synth_pose
    cfg = replace(C1, value_capacity=1 << 13, max_vertices=1 << 21, max_triangles=1 << 22)
    rng = np.random.default_rng(seed)
    pos = np.unique(rng.integers(-spread, spread + 1, size=(count, 3)), axis=0).astype(np.int32)
    vol, orc = Volume(cfg), oracle_mod.Oracle(cfg)
    depth, pose = synth_depth(cfg, 0), synth_pose(cfg, 0)
    vol.upload_depth(depth, pose)
    orc.set_frame(depth, pose)
    triangles = 0
    for step in range(3):
        sdf, weight = _fields(rng, len(pos), cfg)
        vol.load_blocks(pos, sdf, weight)
        orc.load_blocks(pos, sdf, weight)
        if step == 1:  # the blocks in view only
            vol.collect_visible()
            orc.collect_visible()
        else:
            vol.collect_all()
            orc.collect_all()
        assert np.array_equal(vol.dump_candidates(), orc.dump_candidates())
        vol.marching_cubes()
        orc.marching_cubes()
        triangles += _compare(vol, orc)
    assert triangles > 0 or count == 1
    assert vol.status()["flags"] == 0

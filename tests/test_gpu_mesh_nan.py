"""Marching cubes over fields that hold values that are no numbers (a frame with a
broken pose leaves such): a NaN passes the corner tests, as in the reference, and a
vertex on an edge from it has no coordinate that is a number, its normal is zero.
Topology and positions as the oracle has them."""
from dataclasses import replace

import numpy as np
import pytest

from meshhashing_amd.configs import C1
from test_gpu_mesh_blocks import _fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed, share, origin", [(0, 0.002, 0), (1, 0.05, 0), (2, 0.02, 300)])
def test_nan_corners(hip_device, oracle_mod, seed, share, origin):
    from meshhashing_amd.engine import Volume, synth_depth, synth_pose
    cfg = replace(C1, value_capacity=1 << 13, max_vertices=1 << 21, max_triangles=1 << 22)
    rng = np.random.default_rng(seed)
    pos = np.unique(rng.integers(-3, 4, size=(200, 3)), axis=0).astype(np.int32) + np.int32(origin)
    sdf, weight = _fields(rng, len(pos), cfg)
    sdf[rng.random(sdf.shape) < share] = np.nan
    vol, orc = Volume(cfg), oracle_mod.Oracle(cfg)
    vol.upload_depth(synth_depth(cfg, 0), synth_pose(cfg, 0))
    orc.set_frame(synth_depth(cfg, 0), synth_pose(cfg, 0))
    for x in (vol, orc):
        x.load_blocks(pos, sdf, weight)
        x.collect_all()
        x.marching_cubes()
    assert np.array_equal(vol.dump_cube_indices(), orc.dump_blocks()["cube"])
    g, o = vol.dump_mesh(), orc.dump_mesh()
    for k in ("tri_cube", "tri", "vkey", "vref"):
        assert np.array_equal(g[k], o[k]), k
    p = g["vval"][:, :3]
    none = np.isnan(p)
    assert none.any() and np.array_equal(none.any(1), none.all(1))
    assert np.array_equal(p, o["vval"][:, :3].astype(np.float32), equal_nan=True)
    assert not g["vval"][none.any(1), 3:6].any()

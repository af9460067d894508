"""The raycast and its adjoint for poses that are not rigid (a model in other units, a
sheared one): a ray's parameter is then not its camera depth over its direction's, and
no part of it may be left out by the blocks' camera depths.  Against the oracle's plain
march, from beside, inside and far off the blocks."""
from dataclasses import replace

import numpy as np
import pytest

from meshhashing_amd.configs import C1
from test_gpu_raycast_views import _compare, _look

pytestmark = pytest.mark.gpu

SCALES = {"twice": np.diag([2.0, 2.0, 2.0]), "half": np.diag([0.5, 0.5, 0.5]), "axes": np.diag([1.3, 0.7, 2.0]),
          "shear": np.array([[1.0, 0.3, 0.0], [0.0, 1.0, -0.2], [0.1, 0.0, 1.0]]), "mirror": np.diag([-1.0, 1.0, 1.0])}


@pytest.fixture(scope="module")
def blocks(hip_device, oracle_mod):
    from meshhashing_amd.engine import Volume
    cfg = replace(C1, bucket_count=1 << 12, value_capacity=1 << 12)
    rng = np.random.default_rng(7)
    pos = np.unique(rng.integers(-4, 5, size=(400, 3)), axis=0).astype(np.int32)
    i = np.arange(512)
    z = (pos[:, 2:3] * 8 + i // 64) * cfg.voxel_size + (pos[:, 0:1] * 8 + i % 8) * cfg.voxel_size * 0.3
    sdf = (-0.4 * z).astype(np.float32)
    vol, orc = Volume(cfg), oracle_mod.Oracle(cfg)
    for x in (vol, orc):
        x.load_blocks(pos, sdf, np.ones_like(sdf))
    return cfg, vol, orc


@pytest.mark.parametrize("size", [(61, 47), (397, 303), (640, 480)])
@pytest.mark.parametrize("scale", SCALES)
def test_scaled_poses(blocks, scale, size):
    cfg, vol, orc = blocks
    w, h = size
    p = replace(cfg, width=w, height=h, fx=0.82 * w, fy=0.82 * w, cx=0.5 * w, cy=0.5 * h).raycaster_params()
    rng = np.random.default_rng(w)
    S = np.eye(4)
    S[:3, :3] = SCALES[scale]
    hits = []
    for r in (0.2, 0.7, 1.5):
        eye = rng.normal(size=3)
        eye *= r / np.linalg.norm(eye)
        T = (S @ _look(eye, rng.normal(size=3) * 0.1).astype(np.float64)).astype(np.float32)
        hits.append(_compare(cfg, vol, orc, T, p))
        if size == (61, 47):
            import torch
            obs = rng.uniform(0.1, 1.0, w * h).astype(np.float32)
            out = vol.raycast_backward(T, torch.from_numpy(obs).cuda().data_ptr(), params=p)
            ref = orc.raycast_adjoint(False, T, obs, params=p)
            assert out["pixels"] == ref["pixels"]
            assert abs(out["loss"] - ref["loss"]) <= 1e-4 * abs(ref["loss"])
    assert max(hits) > 0  # the views are not empty

"""dL/dsdf against the oracle's adjoint at pixel pitches that fill the wave's
LDS sums differently: many pixels a voxel, about one, and a voxel pitch that no
two pixels share (the table overflows into single atomics)."""
from dataclasses import replace

import numpy as np
import pytest

from meshhashing_amd.configs import C1

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("voxel, size", [(0.04, (8, 8)), (0.04, (320, 240)), (0.01, (37, 29)), (0.01, (160, 120))])
def test_field_gradient_matches_oracle(hip_device, oracle_mod, voxel, size):
    import torch

    from meshhashing_amd.engine import Volume, synth_depth, synth_pose
    w, h = size
    cfg = replace(C1, voxel_size=voxel, truncation=4 * voxel, bucket_count=1 << 15, value_capacity=1 << 14)
    vol = Volume(cfg)
    for f in (2, 3, 4):
        vol.upload_depth(synth_depth(cfg, f), synth_pose(cfg, f))
        vol.alloc()
        vol.collect_visible()
        vol.integrate_tsdf()
    g = vol.dump_blocks()
    orc = oracle_mod.Oracle(cfg)
    orc.load_blocks(g["pos"], g["sdf"], g["weight"], g["color"])
    view = replace(cfg, width=w, height=h, fx=0.82 * w, fy=0.82 * w, cx=0.5 * w, cy=0.5 * h)
    p = view.raycaster_params()
    wTc = synth_pose(cfg, 3).astype(np.float64)
    wTc[:3, 3] += (0.013, -0.009, 0.017)
    cTw = np.linalg.inv(wTc).astype(np.float32)
    obs = np.random.default_rng(w).uniform(1.5, 3.5, w * h).astype(np.float32)
    gs = torch.zeros(cfg.value_capacity * 512, dtype=torch.float32, device=hip_device)
    out = vol.raycast_backward(cTw, torch.from_numpy(obs).to(hip_device).data_ptr(), gs.data_ptr(), params=p)
    ref = orc.raycast_adjoint(False, cTw, obs, params=p, grad_sdf=True)
    assert out["pixels"] == ref["pixels"] > 0
    got = vol.dump_voxel_field(gs.data_ptr())
    # the bar of test_gpu_adjoint: FP32 sums in any order
    assert np.abs(got - ref["grad_sdf"]).max() <= 1e-4 * np.abs(ref["grad_sdf"]).max()

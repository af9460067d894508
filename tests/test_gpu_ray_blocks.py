"""MH_DIAG_RAY_BLOCKS counts the blocks that a raycast's samples lie in, as one
lane a ray takes them: the same number however the image is launched (the tile
shapes other than the first always take one lane a ray), and the count changes
neither the image nor the sample count."""
from dataclasses import replace

import numpy as np
import pytest

from meshhashing_amd import _capi as A
from meshhashing_amd.configs import C1
from meshhashing_amd.engine import Volume, synth_depth, synth_pose

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(8, 8), (61, 47), (160, 120), (352, 263), (640, 480)])
def test_ray_blocks_do_not_depend_on_the_launch(hip_device, size):
    import torch
    cfg = replace(C1, frames=20)
    vol = Volume(cfg)
    for f in (0, 2, 4):
        vol.upload_depth(synth_depth(cfg, f), synth_pose(cfg, f))
        vol.alloc()
        vol.collect_visible()
        vol.integrate_tsdf()
    cTw = vol.pose()[1]
    w, h = size
    p = replace(cfg, width=w, height=h, fx=0.82 * w, fy=0.82 * w, cx=0.5 * w, cy=0.5 * h).raycaster_params()
    d, n = torch.empty(w * h, device=hip_device), torch.empty(3 * w * h, device=hip_device)

    def cast():
        before = vol.status()
        vol.raycast(cTw, d.data_ptr(), 0, n.data_ptr(), params=p)
        after = vol.status()
        return ([after[k] - before[k] for k in ("ray_blocks", "ray_samples")],
                [x.cpu().numpy().view(np.uint32) for x in (d, n)])

    (none, samples), image = cast()
    assert none == 0
    vol.set_diagnostics(ray_blocks=True)
    counts = []
    for shape in range(A.MH_NUM_RAY_SHAPES):
        vol.set_raycast_shape(shape)
        c, im = cast()
        counts.append(c)
        assert all(np.array_equal(a, b) for a, b in zip(im, image))
    assert 0 < counts[0][0] <= vol.status()["block_count"]
    assert counts == [[counts[0][0], samples]] * len(counts)

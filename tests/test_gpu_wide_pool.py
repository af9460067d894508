"""A pool of more than 2^21 blocks, whose voxel fields are over 4 GiB: the raycast,
its adjoint and the localiser address them with 64-bit offsets.  The pool's
first 2^21 slots are taken by blocks far away, so that the scene's blocks lie beyond
4 GiB; what they give is compared with the same scene in a small pool."""
from dataclasses import replace

import numpy as np
import pytest

from meshhashing_amd.configs import C1
from meshhashing_amd.engine import Volume, synth_depth, synth_pose

pytestmark = pytest.mark.gpu

FAR = 1 << 21


def _scene(vol, cfg):
    for f in (2, 3, 4):
        vol.upload_depth(synth_depth(cfg, f), synth_pose(cfg, f))
        vol.alloc()
        vol.collect_visible()
        vol.integrate_tsdf()


@pytest.fixture(scope="module")
def pools(hip_device):
    small = replace(C1, bucket_count=1 << 15, value_capacity=1 << 13)
    large = replace(C1, bucket_count=1 << 20, value_capacity=FAR + (1 << 13))
    wide, narrow = Volume(large), Volume(small)
    chunk = 1 << 17
    far = np.full((chunk, 512), 1.0, np.float32)
    i = np.arange(chunk)
    for k in range(FAR // chunk):  # 128^3 blocks, 320 m away
        pos = np.stack([2000 + 8 * k + i // (128 * 128), i // 128 % 128, i % 128], 1).astype(np.int32)
        wide.load_blocks(pos, far, far)
        print(f"[far blocks] {(k + 1) * chunk}", flush=True)
    assert wide.status()["block_count"] == FAR
    _scene(wide, large)
    _scene(narrow, small)
    st = wide.status(), narrow.status()
    assert st[0]["flags"] == st[1]["flags"] == 0
    assert st[0]["block_count"] - FAR == st[1]["block_count"] > 500
    yield wide, narrow, small
    wide.close()
    narrow.close()


@pytest.mark.parametrize("size", [(61, 47), (352, 263), (640, 480)])
def test_raycast_and_adjoint(pools, size):
    import torch
    wide, narrow, cfg = pools
    w, h = size
    p = replace(cfg, width=w, height=h, fx=0.82 * w, fy=0.82 * w, cx=0.5 * w, cy=0.5 * h).raycaster_params()
    wTc = synth_pose(cfg, 3).astype(np.float64)
    wTc[:3, 3] += (0.013, -0.009, 0.017)
    cTw = np.linalg.inv(wTc).astype(np.float32)
    obs = torch.from_numpy(np.random.default_rng(w).uniform(1.5, 3.5, w * h).astype(np.float32)).cuda()
    image, sums, grad = [], [], []
    for vol in (wide, narrow):
        out = [torch.empty(k * w * h, device="cuda") for k in (1, 3, 3)]
        vol.raycast(cTw, *[x.data_ptr() for x in out], params=p)
        vol.synchronize()
        image.append([x.cpu().numpy().view(np.uint32) for x in out])
        g = torch.zeros(vol.cfg.value_capacity * 512, device="cuda")
        torch.cuda.synchronize()
        sums.append(vol.raycast_backward(cTw, obs.data_ptr(), g.data_ptr(), params=p))
        if vol is wide:
            assert g[:FAR * 512].abs().max() == 0
        grad.append(torch.sort(g[-(512 << 13):])[0].cpu().numpy())
        del g
    assert np.isfinite(image[0][0].view(np.float32)).mean() > 0.5
    for a, b in zip(*image):
        assert np.array_equal(a, b)
    # the same FP64 sums in the same order
    for k in sums[0]:
        assert np.array_equal(sums[0][k], sums[1][k]), k
    # FP32 sums in any order, by value (which slot a block has is a race): the bar of test_gpu_adjoint
    assert np.count_nonzero(grad[1]) > 100
    assert np.abs(grad[0] - grad[1]).max() <= 1e-4 * np.abs(grad[1]).max()


def test_localiser(pools):
    wide, narrow, cfg = pools
    start = synth_pose(cfg, 3).copy()
    start[:3, 3] += [0.01, -0.008, 0.006]
    out = []
    for vol in (wide, narrow):
        vol.upload_depth(synth_depth(cfg, 3), start)
        out.append((vol.point_to_psdf(start, corrected=True), vol.localize(start, iterations=5, lam=1e3, corrected=True)))
    (a, la), (b, lb) = out
    assert a["count"] == b["count"] > 1000
    # FP64 sums of the same terms, by one lane a point and by four
    n = a["count"] * 2.0 ** -52
    for k in ("A", "b", "err"):
        assert np.abs(a[k] - b[k]).max() <= n * max(np.abs(b[k]).max(), np.abs(b["A"]).max())
    assert la["steps"] == lb["steps"] == 5 and np.array_equal(la["count"][:1], lb["count"][:1])
    assert np.abs(la["wTc"] - lb["wTc"]).max() <= 1e-5  # the bar of test_gpu_localize's replay

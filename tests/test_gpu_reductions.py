"""The parallel sums of the adjoint's and the primal-dual energy's partials
at row counts around the reduction's own tile (64 rows)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(8, 8), (8 * 63, 8), (8 * 64, 8), (8 * 65, 8), (8 * 129 - 3, 8 * 33 - 5)])
def test_adjoint_sums_equal_the_raycast_s_residuals(size):
    import torch
    from dataclasses import replace

    from meshhashing_amd.configs import C1
    from meshhashing_amd.engine import Volume, synth_depth, synth_pose

    cfg = replace(C1, frames=20)
    vol = Volume(cfg)
    vol.upload_depth(synth_depth(cfg, 0), synth_pose(cfg, 0))
    vol.alloc()
    vol.collect_visible()
    vol.integrate_tsdf()
    w, h = size
    view = replace(cfg, width=w, height=h, cx=0.5 * w, cy=0.5 * h, fx=262.5, fy=262.5)
    p = view.raycaster_params()
    cTw = vol.pose()[1]
    n = w * h
    d = torch.empty(n, device="cuda")
    vol.raycast(cTw, d.data_ptr(), params=p)
    rng = np.random.default_rng(w)
    obs = rng.uniform(1.0, 4.0, n).astype(np.float32)
    obs[rng.random(n) < 0.1] = 0.0
    out = vol.raycast_backward(cTw, torch.from_numpy(obs).cuda().data_ptr(), params=p, noalloc=True)
    dep = d.cpu().numpy()
    use = np.isfinite(dep) & (obs > 0)
    res = (dep[use] - obs[use]).astype(np.float64)
    assert out["observed"] == int((obs > 0).sum())
    assert out["pixels"] == int(use.sum())
    # two FP64 sums of the same n terms differ by at most n eps of their value
    assert abs(out["loss"] - 0.5 * (res ** 2).sum()) <= n * 2.0 ** -52 * max(out["loss"], 1e-30)


@pytest.mark.parametrize("frames", [1, 6])
def test_energy_on_request_changes_nothing_else(frames):
    from dataclasses import replace

    from meshhashing_amd.configs import C3
    from meshhashing_amd.engine import Volume, synth_depth, synth_pose

    cfg = replace(C3, value_capacity=1 << 16)
    vols = [Volume(cfg) for _ in range(2)]
    for v in vols:
        for f in range(frames):
            v.upload_depth(synth_depth(cfg, f), synth_pose(cfg, f))
            v.alloc()
            v.collect_visible()
            v.predict_inlier()
            v.integrate_psdf()
        v.collect_all()
        v.pd_init()
    for _ in range(3):
        e = vols[0].pd_iterate(0.5, 0.25, 0.25, energy=True)
        vols[1].pd_iterate(0.5, 0.25, 0.25)
    a, b = vols[0].dump_primal_dual(), vols[1].dump_primal_dual()
    for k in a:
        assert np.array_equal(a[k], b[k])
    s = [v.dump_blocks()["sdf"] for v in vols]
    assert np.array_equal(s[0], s[1])
    assert e[0] > 0 and e[1] > 0 and e[2] == e[0] * 0.5 / 2.0 + e[1]

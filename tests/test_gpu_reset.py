"""A volume that was used and reset equals a new one: the same frames give the
same blocks, fields and mesh, also after recycling, after the vertex heap ran
out, and when a caller wrote the pool through a field pointer."""
from dataclasses import replace

import numpy as np
import pytest

from meshhashing_amd.configs import C1, C3

pytestmark = pytest.mark.gpu


def _run(eng, frames):
    from meshhashing_amd.engine import synth_depth, synth_pose
    eng.integrated_frame_count = 0
    for f in frames:
        eng.frame(synth_depth(eng.cfg, f % eng.cfg.frames), synth_pose(eng.cfg, f % eng.cfg.frames))


def _same(a, b):
    for x, y in zip(a, b):
        assert x.keys() == y.keys()
        for k in x:
            assert np.array_equal(x[k], y[k], equal_nan=x[k].dtype.kind == "f"), k


@pytest.mark.parametrize("psdf, verts, held", [(False, 1 << 20, False), (False, 1 << 20, True), (True, 1 << 20, False),
                                               (False, 1 << 13, False)])
def test_reset_volume_equals_a_new_one(hip_device, psdf, verts, held):
    from meshhashing_amd.engine import MainEngine
    base = replace(C3 if psdf else C1, frames=20, max_vertices=verts, value_capacity=(1 << 17) if psdf else 1 << 13)
    used, fresh = MainEngine(base), MainEngine(base)
    if held:
        import torch

        from meshhashing_amd.autograd import sdf_tensor
        sdf_tensor(used.vol).fill_(7.0)
        torch.cuda.synchronize()
        used.vol.reset()
    _run(used, range(0, 16))
    if verts == 1 << 13:
        assert "VERTEX_HEAP_EXHAUSTED" in " ".join(used.vol.status()["flag_names"])
    used.vol.reset()
    st = used.vol.status()
    assert st["block_count"] == st["vertex_count"] == st["triangle_count"] == st["flags"] == 0
    # which vertices an exhausted heap leaves out is a race, and so is what a
    # second frame then frees: one frame, which takes the heap to its end
    frames = [5] if verts == 1 << 13 else [5, 6]
    _run(used, frames)
    _run(fresh, frames)
    a, b = used.vol, fresh.vol
    blocks = a.dump_blocks(), b.dump_blocks()
    _same([blocks[0]], [blocks[1]])
    assert np.array_equal(a.dump_cube_indices(), b.dump_cube_indices())
    if verts != 1 << 13:
        _same([a.dump_mesh()], [b.dump_mesh()])
    else:
        assert a.status()["vertex_count"] == b.status()["vertex_count"]

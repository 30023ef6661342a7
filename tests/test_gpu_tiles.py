"""The tiled force pass on tile lists in run-length order against the lists as built: the same sums in the
same order, so the same bits."""

import numpy as np
import pytest

from test_gpu_plain import build_sim, ctx, host  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile_k,material", [(128, "NH"), (256, "VP"), (512, "MR")])
def test_ordered_tile_lists_change_no_bit(ctx, tile_k, material):  # noqa: F811
    out = []
    for ordered in (True, False):
        sim = build_sim(scatter="tiled", material=material)
        sim.tile_k, sim.fuse_node_pass = tile_k, False
        p = sim.plan()
        assert p.tile_odd == 1 and not p.disp_b
        if not ordered:
            lists = sim.tile_lists(True)
            for k in ("tile_nodes", "tile_lend", "tile_corners", "tile_dst"):
                setattr(p, k, lists[k].data_ptr())
            p.tile_odd = 0
        sim.advance(7)
        out.append((host(sim.displacement, np.float32), host(sim.interactions[-1].velocityB, np.float32)))
    assert np.abs(out[0][0]).max() > 0
    assert all(np.array_equal(a, b) for a, b in zip(*out))


@pytest.mark.parametrize("geo", [True, False])
@pytest.mark.parametrize("material", ["NH", "MR", "VP"])
def test_one_launch_steps_match_two_launch_steps(ctx, material, geo):  # noqa: F811
    """with the shape from the reference positions and with the streamed shape"""
    out = []
    for fuse in (True, False):
        sim = build_sim(scatter="tiled", material=material)
        sim.tile_k, sim.shape_from_ref, sim.fuse_node_pass = 128, geo, fuse
        assert bool(sim.plan().disp_b) == fuse
        sim.advance(120)
        out.append((host(sim.displacement, np.float32), host(sim.interactions[-1].velocityB, np.float32)))
    assert np.abs(out[0][0]).max() > 0
    assert all(np.array_equal(a, b) for a, b in zip(*out))

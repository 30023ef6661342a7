"""GPU test of the batch's one-launch step (the node update of a step inside the next force pass) against its
two-launch step: the same operations in the same order, so positions, velocities, plastic state and curves agree bit
for bit, for calls of one step, two, an odd number, and more than a captured block."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CALLS = (1, 2, 3, 104, 0, 207, 1, 33)
STEPS = sum(CALLS)


@pytest.fixture(scope="module")
def ctx():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from nofluidx3d_amd import openCL

    openCL.initializeOpenCLObjects(0)
    return openCL.handle()


@pytest.mark.parametrize("viscous,kw", [
    (False, {}),
    (False, {"tile_k": 128, "shape_from_ref": False, "narrow": False}),
    (True, {}),
    (True, {"tile_k": 512, "use_graph": False}),
    (True, {"sym_state": False, "plastic_strain": True, "stream_nt": 1}),
])
def test_one_launch_steps_match_two_launch_steps(ctx, monkeypatch, viscous, kw):
    import torch

    from nofluidx3d_amd import autotune
    from nofluidx3d_amd.batch import BatchSimulation, CellSpec, make_meshes

    specs = [CellSpec(2.5 + 0.5 * i, 0.6, 3100 + i, 300.0 * (i + 1), 0.3 + 0.08 * i, 60.0 if viscous else None, 1.0 + i,
                      3.0) for i in range(3)]
    meshes = make_meshes(specs, workers=1, cache=None)

    def run(limit):
        monkeypatch.setattr(autotune, "BATCH_NODE_FUSED_MAX_TETRA", limit)
        b = BatchSimulation(specs, meshes, steps=STEPS, ncurve=50, **kw)
        assert bool(b.plan.disp_b) == (limit > 0)
        for _ in range(2):  # again after a reset
            b.reset(specs)
            for n in CALLS:
                b.advance(n)
            b.sync()
        out = [b.x, b.v, b.curves] + [t for t in (b.state, b.eps, b.t_active) if t is not None]
        return [t.clone() for t in out]

    one, two = run(10 ** 9), run(0)
    assert float(two[2].abs().max()) > 0.0 and bool(torch.isfinite(two[0]).all())
    for s, t in zip(one, two):
        assert np.array_equal(s.cpu().numpy(), t.cpu().numpy())


@pytest.mark.parametrize("tile_k", [128, 256, 512])
def test_curves_do_not_depend_on_the_split_into_calls(ctx, monkeypatch, tile_k):
    """every step is a sample, so every call ends on one, with many nodes in contact: the sum's order is the same in
    a call's last step as inside a call, in both step forms"""
    from nofluidx3d_amd import autotune
    from nofluidx3d_amd.batch import BatchSimulation, CellSpec, make_meshes

    specs = [CellSpec(3.0, 0.3, 3200 + i, 500.0, 0.4, None, 5.0, 3.0, indent_frac=0.5) for i in range(2)]
    meshes = make_meshes(specs, workers=1, cache=None)

    def run(limit, calls):
        monkeypatch.setattr(autotune, "BATCH_NODE_FUSED_MAX_TETRA", limit)
        b = BatchSimulation(specs, meshes, steps=400, ncurve=400, tile_k=tile_k)
        assert bool(b.plan.disp_b) == (limit > 0)
        for n in calls:
            b.advance(n)
        return b.curves_sim()

    whole = run(0, [400])
    assert (whole[:, 200:] > 0).all()
    for limit, calls in ((0, [7] * 57 + [1]), (10 ** 9, [400]), (10 ** 9, [7] * 57 + [1]), (10 ** 9, [2] * 200)):
        assert np.array_equal(run(limit, calls), whole)


@pytest.mark.parametrize("nrep", [1, 2, 3, 8])
def test_timed_passes_are_those_of_the_step_form(ctx, nrep):
    """time_passes on a batch in the node-fused form runs that form (its second buffers are written) from three steps on,
    and advances the batch as the same number of steps does"""
    import torch

    from nofluidx3d_amd.batch import BatchSimulation, CellSpec, make_meshes

    specs = [CellSpec(3.0, 0.5, 3300 + i, 500.0, 0.4, 60.0, 5.0, 3.0, indent_frac=0.5) for i in range(2)]
    meshes = make_meshes(specs, workers=1, cache=None)
    b, want = (BatchSimulation(specs, meshes, steps=100, ncurve=100) for _ in range(2))
    assert b.plan.disp_b
    b.advance(60)
    b.sync()
    before = b.x_b.clone()
    times = b.time_passes(nrep)
    want.advance(60)
    want.advance(nrep)
    for s, t in ((b.x, want.x), (b.v, want.v), (b.state, want.state)):
        assert torch.equal(s, t)
    assert np.array_equal(b.curves_sim(), want.curves_sim()) and b.curves_sim()[:, 59 + nrep].all()
    assert all(t > 0.0 for t in times)
    assert torch.equal(b.x_b, before) == (nrep < 3)

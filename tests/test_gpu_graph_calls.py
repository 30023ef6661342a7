"""GPU test of calls that hold exactly one block of replayed steps: launched by the host at first, captured at the second
call, replayed from then on, and launched step by step while the caller itself captures -- the same bits throughout."""

import ctypes

import numpy as np
import pytest

from test_gpu_plain import build_sim

pytestmark = pytest.mark.gpu

BLOCK = 96


@pytest.fixture(scope="module")
def ctx():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from nofluidx3d_amd import openCL

    openCL.initializeOpenCLObjects(0)
    return openCL.handle()


def captures(h):
    from nofluidx3d_amd import _lib

    n = ctypes.c_int64()
    _lib.call("nfx_graph_captures", h, ctypes.byref(n))
    return n.value


@pytest.mark.parametrize("fuse", [True, False])
@pytest.mark.parametrize("steps,blocks", [(BLOCK + 1, 0), (BLOCK + 3, 1), (2 * BLOCK, 1), (2 * BLOCK + 3, 2)])
def test_call_of_one_block_captures_at_the_second_call(ctx, fuse, steps, blocks):
    def run(use_graph):
        sim = build_sim(scatter="tiled")
        sim.fuse_node_pass, sim.use_graph = fuse, use_graph
        assert bool(sim.plan().disp_b) == fuse
        seen, counts = [], [captures(ctx)]
        for _ in range(4):
            sim.advance(steps)
            counts.append(captures(ctx))
            seen.append((sim.displacement * 1.0).cpu().numpy())
        return seen, np.diff(counts)

    seen, new = run(True)
    assert list(new) == {0: [0, 0, 0, 0], 1: [0, 1, 0, 0], 2: [1, 0, 0, 0]}[blocks]
    ref, none = run(False)
    assert not none.any() and np.abs(ref[-1]).max() > 0
    assert all(np.array_equal(a, b) for a, b in zip(seen, ref))


def test_call_of_one_block_under_the_callers_capture(ctx):
    import torch

    from nofluidx3d_amd import _lib

    side = torch.cuda.Stream()
    h = ctypes.c_void_p()
    _lib.call("nfx_init", 0, side.cuda_stream, ctypes.byref(h))
    sim, ref = build_sim(scatter="tiled"), build_sim(scatter="tiled")
    p = sim.plan()
    torch.cuda.synchronize()
    _lib.call("nfx_run_steps", h, p, 0, 100, None, 1)
    _lib.call("nfx_stream_sync", h)
    n0 = captures(h)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        _lib.call("nfx_run_steps", h, p, 100, 100, None, 1)
    assert captures(h) == n0
    g.replay()
    torch.cuda.synchronize()
    ref.advance(100)
    ref.advance(100)
    assert np.array_equal((sim.displacement * 1.0).cpu().numpy(), (ref.displacement * 1.0).cpu().numpy())
    _lib.call("nfx_destroy", h)


@pytest.mark.parametrize("steps", [20, 120, 2 * BLOCK + 3])
def test_timed_calls_capture_nothing(ctx, steps):
    """the benchmark's timed call and the tuner's, of less than a block of replayed steps, one and two"""
    import bench
    from nofluidx3d_amd import autotune

    assert bench.time_steps(build_sim(scatter="tiled"), 30, steps)[1] == 0
    sim = build_sim(scatter="tiled")
    advance, new = sim.advance, []

    def counted(n):
        before = captures(ctx)
        advance(n)
        new.append(captures(ctx) - before)

    sim.advance = counted
    times = autotune.tune_simulation(sim, nsteps=steps)[1]
    # a candidate's calls: one or two of warm-up, the last one timed
    assert len(new) in (2 * len(times), 3 * len(times))
    assert not any(new[len(new) // len(times) - 1::len(new) // len(times)])

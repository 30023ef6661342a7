"""A context on the default stream, on a stream of its own and on a caller's stream: the same steps, graph
replays with torch work between them included."""

import ctypes

import numpy as np
import pytest

from test_gpu_plain import build_sim, ctx, host  # noqa: F401

pytestmark = pytest.mark.gpu


def test_contexts_on_every_kind_of_stream_step_alike(ctx):  # noqa: F811
    import torch

    from nofluidx3d_amd import _lib

    side = torch.cuda.Stream()
    runs = []
    for stream in (_lib.STREAM_DEFAULT, None, side.cuda_stream):
        h = ctypes.c_void_p()
        _lib.call("nfx_init", 0, stream, ctypes.byref(h))
        sim = build_sim(scatter="tiled")
        p = sim.plan()
        hist = torch.zeros(250, dtype=torch.float64, device="cuda:0")
        seen = []
        for call in range(3):  # 250 steps: two replays of a captured block each
            torch.cuda.synchronize()
            _lib.call("nfx_run_steps", h, p, 250 * call, 250, hist.data_ptr(), 1)
            if stream != _lib.STREAM_DEFAULT:
                _lib.call("nfx_stream_sync", h)  # the default stream's order is torch's own
            seen.append((hist * 1.0).cpu().numpy())
            seen.append((sim.displacement * 1.0).cpu().numpy())
        n = ctypes.c_int64()
        _lib.call("nfx_graph_captures", h, ctypes.byref(n))
        assert n.value == 1
        _lib.call("nfx_destroy", h)
        runs.append(seen)
    assert np.abs(runs[0][-2]).max() > 0
    for other in runs[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(runs[0], other))

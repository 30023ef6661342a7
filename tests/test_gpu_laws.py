"""The elastic laws' Neo-Hookean and Mooney-Rivlin branches at inverted tetra, whose J^-1/3 is NaN (pow() of a
negative number in the reference); their values are held by test_gpu_plain.py."""

import numpy as np
import pytest

from test_gpu_plain import call, ctx, dev, gpu_precompute, host, small_mesh  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ratio", [1.0, 0.75])
def test_inverted_tetra_give_nan_forces(ctx, ratio):  # noqa: F811
    import torch

    from nofluidx3d_amd import _lib

    P, T = small_mesh()
    dminv, v0 = gpu_precompute(ctx, P, T)[:2]
    x = P.copy()
    x[:, 0] *= -1.0  # every tetra mirrored: J = -1
    corners = torch.empty(12 * len(T), dtype=torch.float32, device="cuda:0")
    mat = _lib.Elastic(_lib.NFX_MR, 0.01, 0.45, ratio)
    xd, td = dev(x.reshape(-1, order="F"), np.float32), dev(T.reshape(-1, order="F").astype(np.uint32))
    call("nfx_tetra_corner_forces", ctx, mat, xd.data_ptr(), td.data_ptr(), dminv.data_ptr(), v0.data_ptr(), len(P),
         len(T), corners.data_ptr())
    assert np.isnan(host(corners)).all()

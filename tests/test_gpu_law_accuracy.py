"""Rounding error of the elastic laws' corner forces against float64, where a form of the law can lose it: large rotations
with little strain or none, and tetra compressed to a fraction of their volume.  The measure is the error of the spatial
form -- B - I and J - 1 from the displacement gradient, sigma, cof(F) -- with every operation rounded once to float32 and
J^-1/3 from a logarithm and an exponential of 1 ulp: the law may be at most half again as far off (root mean square
over the tetra), a margin for another order of its sums."""

import numpy as np
import pytest

from test_gpu_plain import call, ctx, dev, host  # noqa: F401

pytestmark = pytest.mark.gpu

E, COUNT = 0.01, 20000
f32 = np.float32


def rotations(rng, angle):
    a = rng.normal(size=(COUNT, 3))
    x, y, z = (a / np.linalg.norm(a, axis=1)[:, None]).T
    o = np.zeros(COUNT)
    K = np.array([[o, -z, y], [z, o, -x], [-y, x, o]]).transpose(2, 0, 1)
    return np.eye(3) + np.sin(angle) * K + (1 - np.cos(angle)) * (K @ K)


def deformations(kind, size, rng):
    if kind == "rotation":
        return rotations(rng, size)
    if kind == "strain":  # under a rotation by 0.1
        A = rng.uniform(-1, 1, (COUNT, 3, 3))
        return rotations(rng, 0.1) @ (np.eye(3) + 0.5 * size * (A + A.transpose(0, 2, 1)))
    R, s = rotations(rng, 1.0), rng.uniform(size, size + 0.1, (COUNT, 3))  # principal stretches from size on
    return rotations(rng, 0.3) @ R @ (s[:, :, None] * R.transpose(0, 2, 1))


def spatial_form(H, mu1, mu2, kappa, rng=None):
    """sigma cof(F) in the precision of H; rng: errors of up to 1 ulp of the logarithm and of the exponential."""
    t = H.dtype.type
    det = lambda A: (A[:, 0, 0] * (A[:, 1, 1] * A[:, 2, 2] - A[:, 1, 2] * A[:, 2, 1])
                     - A[:, 0, 1] * (A[:, 1, 0] * A[:, 2, 2] - A[:, 1, 2] * A[:, 2, 0])
                     + A[:, 0, 2] * (A[:, 1, 0] * A[:, 2, 1] - A[:, 1, 1] * A[:, 2, 0]))
    minor = lambda i, j: H[:, i, i] * H[:, j, j] - H[:, i, j] * H[:, j, i]
    mul = lambda A, B: A[:, :, 0, None] * B[:, None, 0] + A[:, :, 1, None] * B[:, None, 1] + A[:, :, 2, None] * B[:, None, 2]
    tr = lambda A: A[:, 0, 0] + A[:, 1, 1] + A[:, 2, 2]
    I = np.eye(3, dtype=t)
    dev3 = lambda A: A - (tr(A) * t(1 / 3))[:, None, None] * I
    c = lambda v: np.asarray(v, t)[..., None, None]
    ulp = lambda v: v if rng is None else (v * (1 + rng.uniform(-1, 1, v.shape) * 2.0 ** -23)).astype(t)
    HT = H.transpose(0, 2, 1)
    Bd = (H + HT) + mul(H, HT)
    Jm1 = tr(H) + ((minor(0, 1) + minor(0, 2) + minor(1, 2)) + det(H))
    p = ulp(np.exp2(ulp(np.log2(t(1) + Jm1)) * t(-1 / 3)))
    p2 = p * p
    p5 = p2 * p2 * p
    a, k = t(mu1) * p5, t(mu2) * p5 * p2
    sig = c(a + k) * dev3(Bd) + c(t(kappa) * Jm1) * I
    if mu2:
        sig = sig + c(k) * dev3(c(tr(Bd)) * Bd - mul(Bd, Bd))
    F = H + I
    cross = lambda u, v: np.stack([u[:, 1] * v[:, 2] - u[:, 2] * v[:, 1], u[:, 2] * v[:, 0] - u[:, 0] * v[:, 2],
                                   u[:, 0] * v[:, 1] - u[:, 1] * v[:, 0]], 1)
    cof = np.stack([cross(F[:, 1], F[:, 2]), cross(F[:, 2], F[:, 0]), cross(F[:, 0], F[:, 1])], 1)
    return mul(sig, cof)


@pytest.mark.parametrize("nu", [0.0, 0.3])
@pytest.mark.parametrize("ratio,kind,size", [
    (1.0, "rotation", 0.01), (1.0, "rotation", 0.03), (1.0, "strain", 0.001), (1.0, "strain", 0.1),
    (1.0, "stretch", 0.5), (1.0, "stretch", 0.9),
    (0.75, "rotation", 0.03), (0.75, "strain", 0.1), (0.75, "stretch", 0.5), (0.25, "stretch", 0.6), (0.25, "stretch", 0.9),
])
def test_law_rounds_no_more_than_its_spatial_form(ctx, nu, ratio, kind, size):  # noqa: F811
    import torch

    from nofluidx3d_amd import _lib

    rng = np.random.default_rng(7)
    x = deformations(kind, size, rng).transpose(0, 2, 1).astype(f32)  # rows: the three edges from a corner at 0
    mu = E / (2 * (1 + nu))
    consts = [float(f32(v)) for v in (ratio * mu, (1 - ratio) * mu, E / (3 * (1 - 2 * nu)))]
    H = x.transpose(0, 2, 1) - np.eye(3, dtype=f32)  # as the kernel forms it: the edges times I, less I
    ref = spatial_form(H.astype(np.float64), *consts)
    norm = np.linalg.norm(ref, axis=(1, 2)) if kind != "rotation" else mu
    rms = lambda P: np.sqrt(np.mean((np.linalg.norm(P - ref, axis=(1, 2)) / norm) ** 2))

    pts = np.concatenate([np.zeros((COUNT, 1, 3), f32), x], 1).reshape(-1, 3)
    tets = np.arange(4 * COUNT, dtype=np.uint32).reshape(-1, 4)
    dminv = np.repeat(np.eye(3, dtype=f32).reshape(9, 1), COUNT, 1)
    corners = torch.empty(12 * COUNT, dtype=torch.float32, device="cuda:0")
    mat = _lib.Elastic(_lib.NFX_MR, E, nu, ratio)
    ins = [dev(pts.reshape(-1, order="F"), f32), dev(tets.reshape(-1, order="F")), dev(dminv.reshape(-1), f32),
           dev(np.full(COUNT, 1 / 6), f32)]
    call("nfx_tetra_corner_forces", ctx, mat, *[t.data_ptr() for t in ins], 4 * COUNT, COUNT, corners.data_ptr())
    f = host(corners, f32).astype(np.float64).reshape(COUNT, 4, 3)
    got, allowed = rms(-6.0 * f[:, 1:].transpose(0, 2, 1)), 1.5 * rms(spatial_form(H, *consts, rng=rng))
    assert got <= allowed, (got, allowed)

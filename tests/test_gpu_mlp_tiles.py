"""GPU tests of the edges of the MLP kernels' tiles, k-steps and wide accesses.

The GEMM operands are small whole numbers, whose products and sums are exact in FP32: results equal the integer
product.  The loss gradient and its transpose are compared bit for bit with the same FP32 expression; the loss within
1e-12 and the bias sums within 6e-6 of FP64 (a thread adds at most 16 entries below 1/16, a tree of 8 levels the
rest: at most 24 roundings of sums below 4, 24 * 4 * 2^-24 < 6e-6).
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from nofluidx3d_amd import openCL

    openCL.initializeOpenCLObjects(0)
    return openCL.handle()


def shifted(n, dtype, off):
    """A device vector of n entries that starts ``off`` entries into its allocation."""
    import torch

    return torch.zeros(n + off, dtype=dtype, device="cuda:0")[off:]


# k-steps of 32 (K / S no multiple of 64) and of 64, one step and several, one column tile and several, K slices of
# each kind, operands with longer rows, the transposed copy at 8-byte and at 2-byte alignment
@pytest.mark.parametrize("M,N,K,S,pad,off", [(128, 32, 32, 1, 0, 0), (128, 32, 96, 1, 8, 1), (128, 96, 64, 1, 0, 3),
                                             (384, 64, 192, 1, 24, 0), (256, 64, 96, 3, 0, 2), (128, 160, 448, 7, 8, 0),
                                             (32768, 128, 64, 1, 0, 1), (33024, 512, 32, 1, 8, 0),
                                             (65536, 256, 96, 1, 0, 0)])
def test_gemm_of_whole_numbers_is_exact(ctx, M, N, K, S, pad, off):
    import torch

    from nofluidx3d_amd import _lib
    from nofluidx3d_amd.surrogate.mlp import MLP

    rng = np.random.default_rng(M + N + K)
    a, b = rng.integers(-3, 4, (M, K + pad)), rng.integers(-3, 4, (N, K + pad))
    A, B = (torch.tensor(x, dtype=torch.float32).to(torch.bfloat16).cuda() for x in (a, b))
    ref = a[:, :K] @ b[:, :K].T
    ws = torch.empty(S * M * N, dtype=torch.float32, device="cuda:0") if S > 1 else None
    C = torch.empty(M, N, dtype=torch.float32, device="cuda:0")
    MLP._gemm(_lib.NFX_MLP_STORE, M, N, K, A, K + pad, B, K + pad, C=C, split=S, ws=ws)
    assert np.array_equal(C.cpu().numpy(), ref)
    bias = torch.zeros(N, dtype=torch.float32, device="cuda:0")
    H = torch.empty(M, N, dtype=torch.bfloat16, device="cuda:0")
    HT = shifted(N * M, torch.bfloat16, off).view(N, M)
    MLP._gemm(_lib.NFX_MLP_FWD_GELU, M, N, K, A, K + pad, B, K + pad, bias=bias, C=C, H=H, HT=HT, split=S, ws=ws)
    assert np.array_equal(C.cpu().numpy(), ref)
    assert torch.equal(H.t().contiguous(), HT)
    # the gradient epilogue at Z = 0 halves the product
    dT = shifted(N * M, torch.bfloat16, off).view(N, M)
    MLP._gemm(_lib.NFX_MLP_BWD_GELU, M, N, K, A, K + pad, B, K + pad, Z=torch.zeros_like(C), H=H, HT=dT, split=S, ws=ws)
    assert torch.equal(H.cpu(), (torch.tensor(ref, dtype=torch.float32) * 0.5).to(torch.bfloat16))
    assert torch.equal(H.t().contiguous(), dT)


@pytest.mark.parametrize("M,N,weighted", [(32, 32, False), (96, 64, True), (128, 32, True), (384, 96, False)])
def test_mse_tiles(ctx, M, N, weighted):
    import torch

    from nofluidx3d_amd import _lib

    g = torch.Generator().manual_seed(M + N)
    Y, T = torch.randn(M, N, generator=g), torch.randn(M, N, generator=g)
    w = torch.rand(M, generator=g) if weighted else None
    dev = [None if x is None else x.cuda() for x in (Y, T, w)]
    dZ = torch.empty(M, N, dtype=torch.bfloat16, device="cuda:0")
    dZT = torch.empty(N, M, dtype=torch.bfloat16, device="cuda:0")
    loss = torch.zeros(1, dtype=torch.float64, device="cuda:0")
    _lib.call("nfx_mlp_mse", ctx, dev[0].data_ptr(), dev[1].data_ptr(), dev[2].data_ptr() if weighted else None, M, N,
              dZ.data_ptr(), dZT.data_ptr(), loss.data_ptr())
    wr = torch.ones(M) if w is None else w
    d = Y - T
    sc = np.float32(2.0) / (np.float32(M) * np.float32(N))
    assert torch.equal(dZ.cpu(), ((float(sc) * wr)[:, None] * d).to(torch.bfloat16))
    assert torch.equal(dZ.t().contiguous(), dZT)
    ref = float((wr.double()[:, None] * d.double() * d.double()).sum()) / (M * N)
    assert abs(float(loss) - ref) <= 1e-12 * ref


@pytest.mark.parametrize("M,off", [(1, 0), (1001, 0), (1000, 0), (1000, 1), (4096, 0), (8, 0)])
def test_bias_sums(ctx, M, off):
    import torch

    from nofluidx3d_amd import _lib

    N = 5
    z = (torch.rand(N, M, generator=torch.Generator().manual_seed(M)) * 2 - 1).div(16).to(torch.bfloat16)
    dZT = shifted(N * M, torch.bfloat16, off)
    dZT.copy_(z.reshape(-1))
    b, m, v = (torch.zeros(N, dtype=torch.float32, device="cuda:0") for _ in range(3))
    # beta1 = 0: the first moment is the row sum
    _lib.call("nfx_mlp_bias_adam", ctx, dZT.data_ptr(), M, N, b.data_ptr(), m.data_ptr(), v.data_ptr(), 1e-3, 1.0, 0.0,
              0.0, 1e-8, 1.0)
    ref = z.double().sum(1).numpy()
    assert np.max(np.abs(m.cpu().numpy() - ref)) <= 6e-6
    assert np.allclose(b.cpu().numpy(), -1e-3 * ref / (np.abs(ref) + 1e-8), rtol=1e-5, atol=0)

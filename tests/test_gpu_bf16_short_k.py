"""Short sums over many tiles on the eight-wave 128x128 BF16 tile (GPU): the
two-buffer form up to its limit (128 k split, 256 single BF16) and the
four-buffer form past it, full and triangular, against FP64. Bar: relative
Frobenius error on U[-1, 1) inputs, 1e-5 (split) or 1e-2 (single BF16)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = {"split-bf16": 1e-5, "bf16": 1e-2}


def seeded(h, rows, cols, mid):
    x = torch.empty((rows, cols), device=DEV)
    h.fill_uniform(x, 23, mid)
    return x


@pytest.mark.parametrize("prec", ["split-bf16", "bf16"])
@pytest.mark.parametrize("k", [1, 32, 79, 128, 129, 256, 257])
def test_short_k(handle, mfx, prec, k):
    print(f"short k {prec} {k}", flush=True)
    m, n = 2101, 2070  # 17 x 17 tiles
    A, B, C0 = seeded(handle, m, k, 0), seeded(handle, k, n, 1), seeded(handle, m, n, 2)
    S0 = seeded(handle, 3000, 3000, 3)  # a triangle of 300 tiles
    L = seeded(handle, 3000, k, 4)
    handle.force_config(prec, 6)
    try:
        C, S = C0.clone(), S0.clone()
        handle.gemm(A, B, C, alpha=1.5, beta=0.5, prec=prec)
        handle.syrk(L, S, alpha=1.5, beta=0.5, prec=prec, uplo=mfx.LOWER, mirror=False)
    finally:
        handle.force_config(prec, -1)
    want = 1.5 * (A.double() @ B.double()) + 0.5 * C0.double()
    assert torch.linalg.norm(C.double() - want) < TOL[prec] * torch.linalg.norm(want)
    want = torch.tril(1.5 * (L.double() @ L.double().T) + 0.5 * S0.double())
    assert torch.linalg.norm(torch.tril(S).double() - want) < TOL[prec] * torch.linalg.norm(want)
    assert torch.equal(torch.triu(S, 1), torch.triu(S0, 1))

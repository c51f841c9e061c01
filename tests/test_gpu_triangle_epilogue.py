"""Triangle stores (GPU): interior, diagonal and edge blocks, with C rows that
16-byte stores fit and that they do not, mirrored and not, old values used and
not.  Bar: relative Frobenius error against FP64 on U[-1, 1) inputs, 2e-6
(FP32) or 1e-5 (split BF16); a symmetric C stays symmetric to the last bit, and
what lies outside the triangle stays untouched without `mirror`."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = {"fp32": 2e-6, "split-bf16": 1e-5}


@pytest.mark.parametrize("prec", ["fp32", "split-bf16"])
@pytest.mark.parametrize("n", [31, 64, 97, 260, 700])
@pytest.mark.parametrize("pad", [0, 1, 4])
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_triangle_blocks(handle, mfx, prec, n, pad, beta):
    print(f"triangle {prec} {n} pad {pad} beta {beta}", flush=True)
    k = 96
    A = torch.empty((n, k), device=DEV)
    C0 = torch.empty((n, n), device=DEV)
    handle.fill_uniform(A, 5, 0)
    handle.fill_uniform(C0, 5, 1)
    C0 = torch.tril(C0) + torch.tril(C0, -1).T
    want = 1.5 * (A.double() @ A.double().T) + beta * C0.double()
    for uplo in (mfx.LOWER, mfx.UPPER):
        for mirror in (True, False):
            C = torch.full((n, n + pad), 7.0, device=DEV)
            C[:, :n] = C0
            handle.syrk(A, C[:, :n], alpha=1.5, beta=beta, prec=prec, uplo=uplo, mirror=mirror)
            got = C[:, :n]
            assert torch.equal(C[:, n:], torch.full((n, pad), 7.0, device=DEV))
            inside = torch.tril if uplo == mfx.LOWER else torch.triu
            err = torch.linalg.norm(inside(got.double() - want)) / torch.linalg.norm(inside(want))
            assert err < TOL[prec]
            if mirror:
                assert torch.equal(got, got.T)
            else:
                assert torch.equal(got - inside(got), C0 - inside(C0))

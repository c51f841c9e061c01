"""Edges of the FP32 tile (GPU, through the C ABI): partial last stages of
every length class, operand layouts, 16-byte and 4-byte copies, tiles past
the matrix, two products, slices of full and triangular schedules.

Operands sit in rows padded with NaN, so any value read from beyond K or a
row's end shows.  Bar: relative Frobenius error 2e-6 against FP64 on
U[-1, 1) inputs (the FP32 method's bar; four times that below 16 k, where one
rounding is a larger share of the norm)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = 2e-6


def seeded(h, rows, cols, mid, pad):
    base = torch.full((rows, cols + pad), float("nan"), device=DEV)
    x = torch.empty((rows, cols), device=DEV)
    h.fill_uniform(x, 13, mid)
    base[:, :cols] = x
    return base[:, :cols]


def rel(got, want, mask=None):
    d, w = got.double() - want, want
    if mask is not None:
        d, w = d[mask], w[mask]
    return (torch.linalg.norm(d) / torch.linalg.norm(w)).item()


@pytest.mark.parametrize("config", range(8))
@pytest.mark.parametrize("k", [1, 4, 15, 16, 20, 31, 33, 64, 100])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_k_tails(handle, config, k, ta, tb):
    handle.force_config("fp32", config)
    try:
        # pad 4: 16-byte rows where the contiguous extent allows; pad 3: 4-byte copies
        for m, n, pad in ((68, 36, 4), (70, 261, 3)):
            print(f"config {config} {m}x{n}x{k} ta={ta} tb={tb} pad={pad}", flush=True)
            A = seeded(handle, k if ta else m, m if ta else k, 0, pad)
            B = seeded(handle, n if tb else k, k if tb else n, 1, pad)
            C = torch.full((m, n + pad), float("nan"), device=DEV)[:, :n]
            for splits in (1, 3):
                handle.force_splits(splits)
                handle.gemm(A, B, C, alpha=1.5, beta=0.0, prec="fp32", transA=ta, transB=tb)
                want = 1.5 * (A.double().T if ta else A.double()) @ (B.double().T if tb else B.double())
                assert rel(C, want) < (TOL if k >= 16 else 4 * TOL), splits
                assert torch.isnan(C.as_strided((m, pad), (n + pad, 1), n)).all()
    finally:
        handle.force_config("fp32", -1)
        handle.force_splits(-1)


@pytest.mark.parametrize("config", [0, 1, 4, 6, 7])
@pytest.mark.parametrize("splits", [1, 4])
@pytest.mark.parametrize("uplo,mirror", [(0, True), (1, True), (0, False), (1, False)])
@pytest.mark.parametrize("n,k,pad", [(300, 200, 4), (131, 77, 3)])
def test_triangles_one_and_two_products(handle, config, splits, uplo, mirror, n, k, pad):
    print(f"config {config} n={n} k={k} uplo={uplo} mirror={mirror} S={splits}", flush=True)
    A, B = seeded(handle, n, k, 0, pad), seeded(handle, n, k, 1, pad)
    C0 = torch.empty((n, n), device=DEV)
    handle.fill_uniform(C0, 13, 2)
    A64, B64 = A.double(), B.double()
    ones = torch.ones((n, n), dtype=torch.bool, device=DEV)
    mask = ones if mirror else ones.tril() if uplo == 0 else ones.triu()
    handle.force_config("fp32", config)
    handle.force_splits(splits)
    try:
        for which, P in (("syrk", A64 @ A64.T), ("syr2k", A64 @ B64.T + B64 @ A64.T)):
            C = C0.clone()
            if which == "syrk":
                handle.syrk(A, C, alpha=0.75, beta=1.25, prec="fp32", uplo=uplo, mirror=mirror)
            else:
                handle.syr2k(A, B, C, alpha=0.75, beta=1.25, prec="fp32", uplo=uplo, mirror=mirror)
            assert rel(C, 0.75 * P + 1.25 * C0.double(), mask) < TOL, which
            assert torch.equal(C[~mask], C0[~mask])
    finally:
        handle.force_config("fp32", -1)
        handle.force_splits(-1)

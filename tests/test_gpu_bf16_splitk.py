"""Split-K of the packed BF16 and FP8 paths (GPU, through the C ABI):
whole tiles and k slices in one launch, the slices' partial tiles summed in
slice order by splitk_reduce, on full and triangular schedules.

Bars: relative Frobenius error against FP64 on U[-1, 1) inputs at the
precision's tolerance (1e-5 split, 1e-2 single BF16: the rounding of the
operands, which splitting does not touch), elements outside the requested
triangle untouched, beta = 0 never reads C, repeated calls bit-identical.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = {"split-bf16": 1e-5, "bf16": 1e-2}


def seeded(h, rows, cols, mid, pad=0):
    base = torch.empty((rows, cols + pad), device=DEV)
    x = base[:, :cols]
    h.fill_uniform(x, 5, mid)
    return x


def rel(got, want, mask=None):
    d, w = got.double() - want, want
    if mask is not None:
        d, w = d[mask], w[mask]
    return (torch.linalg.norm(d) / torch.linalg.norm(w)).item()


def recorded(h, call):
    h.timing_begin()
    call()
    rec = h.timing_end()
    torch.cuda.synchronize()
    return rec


@pytest.mark.parametrize("prec", ["split-bf16", "bf16"])
@pytest.mark.parametrize("config", [0, 1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("m,n,k,ta,tb,pad,splits", [
    (64, 64, 2048, False, False, 0, 8),      # one small tile
    (300, 517, 1000, True, True, 4, 3),      # ragged tiles, padded rows, k off the stage
    (33, 70, 130, False, True, 3, 5),        # unaligned rows, slices of one stage
    (257, 255, 96, True, False, 0, 64),      # fewer stages than slices
])
def test_forced_splits_every_tile(handle, prec, config, m, n, k, ta, tb, pad, splits):
    print(f"split {prec} config {config} {m}x{n}x{k} ta={ta} tb={tb} pad={pad} S={splits}", flush=True)
    A = seeded(handle, k if ta else m, m if ta else k, 0, pad)
    B = seeded(handle, n if tb else k, k if tb else n, 1, pad)
    C0 = seeded(handle, m, n, 2, pad)
    want = 1.5 * (A.double().T if ta else A.double()) @ (B.double().T if tb else B.double())
    handle.force_config(prec, config)
    handle.force_splits(splits)
    try:
        for beta in (1.2, 0.0):
            outs = []
            for _ in range(2):
                C = torch.full((m, n + pad), float("nan"), device=DEV)[:, :n]
                if beta:
                    C.copy_(C0)
                rec = recorded(handle, lambda: handle.gemm(A, B, C, alpha=1.5, beta=beta, prec=prec, transA=ta, transB=tb))
                outs.append(C)
            assert "splitk_reduce" in rec, rec
            assert torch.equal(outs[0], outs[1])
            ref = want + beta * C0.double() if beta else want
            assert rel(outs[0], ref) < TOL[prec]
            if pad:  # the padding columns are not written
                assert torch.isnan(outs[0].as_strided((m, pad), (n + pad, 1), n)).all()
    finally:
        handle.force_config(prec, -1)
        handle.force_splits(-1)


@pytest.mark.parametrize("prec", ["split-bf16", "bf16"])
@pytest.mark.parametrize("uplo,mirror", [(0, False), (0, True), (1, False), (1, True), (2, False)])
@pytest.mark.parametrize("n,k,config", [(70, 300, 2), (300, 1000, 6), (513, 260, 4)])
def test_triangles(handle, prec, uplo, mirror, n, k, config):
    print(f"split triangle {prec} uplo={uplo} mirror={mirror} n={n} k={k} config={config}", flush=True)
    A, B, C0 = seeded(handle, n, k, 0), seeded(handle, n, k, 1), seeded(handle, n, n, 2)
    A64, B64 = A.double(), B.double()
    prods = {"syrk": A64 @ A64.T, "syr2k": A64 @ B64.T + B64 @ A64.T}
    ones = torch.ones((n, n), dtype=torch.bool, device=DEV)
    mask = ones if mirror or uplo == 2 else ones.tril() if uplo == 0 else ones.triu()
    handle.force_config(prec, config)
    handle.force_splits(3)
    try:
        for which, P in prods.items():
            C = C0.clone()
            if which == "syrk":
                rec = recorded(handle, lambda: handle.syrk(A, C, alpha=0.75, beta=1.25, prec=prec, uplo=uplo, mirror=mirror))
            else:
                rec = recorded(handle, lambda: handle.syr2k(A, B, C, alpha=0.75, beta=1.25, prec=prec, uplo=uplo,
                                                            mirror=mirror))
            assert "splitk_reduce" in rec, rec
            assert rel(C, 0.75 * P + 1.25 * C0.double(), mask) < TOL[prec], which
            assert torch.equal(C[~mask], C0[~mask])
    finally:
        handle.force_config(prec, -1)
        handle.force_splits(-1)


@pytest.mark.parametrize("prec", ["split-bf16", "bf16"])
def test_whole_rounds_and_a_split_rest(handle, prec):
    """One round of whole 128x128 tiles (one per CU) and a few tiles beyond it, which split."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    m, n, k = 128 * 8, 128 * (cus // 8 + 1) - 3, 2048
    print(f"whole round + rest {prec} {m}x{n}x{k}", flush=True)
    A, B, C0 = seeded(handle, m, k, 0), seeded(handle, k, n, 1), seeded(handle, m, n, 2)
    C = C0.clone()
    handle.force_config(prec, 6)
    try:
        rec = recorded(handle, lambda: handle.gemm(A, B, C, alpha=1.5, beta=0.5, prec=prec))
    finally:
        handle.force_config(prec, -1)
    assert "splitk_reduce" in rec, rec
    assert rel(C, 1.5 * A.double() @ B.double() + 0.5 * C0.double()) < TOL[prec]


@pytest.mark.parametrize("prec", ["fp8-block", "fp8-block2"])
@pytest.mark.parametrize("config", [0, 1, 2, 3])
@pytest.mark.parametrize("m,n,k,ta,tb,splits", [(64, 64, 128, False, False, 2), (200, 130, 700, True, False, 3),
                                                (300, 270, 1000, False, True, 64)])
def test_fp8_slices(handle, prec, config, m, n, k, ta, tb, splits):
    """Slices of block-scaled FP8 tiles against the whole tiles' result: the
    same codes and scales, so they differ by the instruction's summation error
    only (about 2^-15 relative per 64-wide dot, as for the product itself)."""
    print(f"fp8 split {prec} config {config} {m}x{n}x{k} ta={ta} tb={tb} S={splits}", flush=True)
    A = seeded(handle, k if ta else m, m if ta else k, 0)
    B = seeded(handle, n if tb else k, k if tb else n, 1)
    C0 = seeded(handle, m, n, 2)
    outs = {}
    handle.force_config(prec, config)
    try:
        for s in (1, splits):
            handle.force_splits(s)
            C = C0.clone()
            rec = recorded(handle, lambda: handle.gemm(A, B, C, alpha=1.5, beta=0.5, prec=prec, transA=ta, transB=tb))
            assert ("splitk_reduce" in rec) == (s > 1 and k > 128), rec
            outs[s] = C
    finally:
        handle.force_config(prec, -1)
        handle.force_splits(-1)
    assert rel(outs[splits], outs[1].double()) < 1e-4

"""Launches that mix whole tiles with k slices (GPU, through the C ABI): tiles
of 128x128 that fill one round of the CUs and a few more, which run as slices,
on full grids (FP32, FP8) and triangles. The tiles of the whole round are bit
for bit those of an unsplit launch; the result keeps the precision's bar against
FP64 (relative Frobenius error 2e-6 FP32, 1e-5 split and 1e-2 single BF16), FP8
that of its unsplit result (1e-4: the same codes, another order of sums). And
which form of the eight-wave BF16 tile short sums take."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = {"fp32": 2e-6, "split-bf16": 1e-5, "bf16": 1e-2}


def seeded(h, rows, cols, mid):
    x = torch.empty((rows, cols), device=DEV)
    h.fill_uniform(x, 41, mid)
    return x


def both(h, prec, config, call, C0):
    """The call's result with automatic slices and with none, and the kernels of the first."""
    out = {}
    h.force_config(prec, config)
    try:
        for splits in (-1, 1):
            h.force_splits(splits)
            C = C0.clone()
            h.timing_begin()
            call(C)
            rec = h.timing_end()
            assert ("splitk_reduce" in rec) == (splits < 0), rec
            out[splits] = C
    finally:
        h.force_config(prec, -1)
        h.force_splits(-1)
    return out[-1], out[1]


def equal_tiles(a, b, wanted):
    """Of the 128x128 tiles that hold wanted elements, how many are the same bits, and how many there are."""
    same = total = 0
    for i in range(0, a.shape[0], 128):
        for j in range(0, a.shape[1], 128):
            w = wanted[i:i + 128, j:j + 128]
            if bool(w.any()):
                total += 1
                same += torch.equal(a[i:i + 128, j:j + 128][w], b[i:i + 128, j:j + 128][w])
    return same, total


@pytest.fixture
def cus():
    n = torch.cuda.get_device_properties(0).multi_processor_count
    if n != 256:
        pytest.skip("sizes are for 256 CUs")
    return n


@pytest.mark.parametrize("prec,config", [("fp32", 6), ("fp8-block", 1), ("fp8-block2", 1)])
def test_full_grid(handle, cus, prec, config):
    m, n, k = 128 * 8, 128 * (cus // 8 + 1) - 3, 4096
    print(f"mixed rounds {prec} {m}x{n}x{k}", flush=True)
    A, B, C0 = seeded(handle, m, k, 0), seeded(handle, k, n, 1), seeded(handle, m, n, 2)
    got, whole = both(handle, prec, config, lambda C: handle.gemm(A, B, C, alpha=1.5, beta=0.5, prec=prec), C0)
    same, total = equal_tiles(got, whole, torch.ones_like(C0, dtype=torch.bool))
    assert total == cus + 8 and cus <= same < total, (same, total)
    want = whole.double() if prec.startswith("fp8") else 1.5 * A.double() @ B.double() + 0.5 * C0.double()
    assert torch.linalg.norm(got.double() - want) < TOL.get(prec, 1e-4) * torch.linalg.norm(want)


@pytest.mark.parametrize("prec", ["fp32", "split-bf16", "bf16"])
@pytest.mark.parametrize("kind,k", [("syrk", 4096), ("syr2k", 2048)])
@pytest.mark.parametrize("uplo,mirror", [(0, False), (0, True), (1, False), (1, True)])
def test_triangle(handle, cus, prec, kind, k, uplo, mirror):
    n = 3000  # 300 tiles
    print(f"mixed rounds {kind} {prec} n={n} k={k} uplo={uplo} mirror={mirror}", flush=True)
    A, B, C0 = seeded(handle, n, k, 0), seeded(handle, n, k, 1), seeded(handle, n, n, 2)
    P = A.double() @ (A if kind == "syrk" else B).double().T
    P = P if kind == "syrk" else P + P.T
    opt = dict(alpha=0.75, beta=1.25, prec=prec, uplo=uplo, mirror=mirror)
    call = (lambda C: handle.syrk(A, C, **opt)) if kind == "syrk" else (lambda C: handle.syr2k(A, B, C, **opt))
    got, whole = both(handle, prec, 6, call, C0)
    ones = torch.ones((n, n), dtype=torch.bool, device=DEV)
    half = ones.tril() if uplo == 0 else ones.triu()
    same, total = equal_tiles(got, whole, half)
    assert total == 300 and cus <= same < total, (same, total)
    mask = ones if mirror else half
    want = 0.75 * P + 1.25 * C0.double()
    assert torch.linalg.norm((got.double() - want)[mask]) < TOL[prec] * torch.linalg.norm(want[mask])
    assert torch.equal(got[~mask], C0[~mask])


@pytest.mark.parametrize("prec,name,most", [("split-bf16", "gemm_split_bf16", 128), ("bf16", "gemm_bf16", 256)])
def test_short_sums_take_two_buffers(handle, cus, prec, name, most):
    for k in (most - 1, most, most + 1):
        A, B, C = seeded(handle, 2101, k, 0), seeded(handle, k, 2070, 1), torch.empty((2101, 2070), device=DEV)
        handle.force_config(prec, 6)
        handle.timing_begin()
        try:
            handle.gemm(A, B, C, prec=prec)
        finally:
            handle.force_config(prec, -1)
        rec = handle.timing_end()
        assert (name + "_short_k" in rec) == (k <= most) and (name + "_mfma" in rec) == (k > most), (k, rec)

"""Short lists under a loaded or measured tuning table (GPU, through the C ABI)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = {"fp32": 2e-6, "split-bf16": 1e-5, "bf16": 1e-2}


@pytest.fixture
def table(mfx, tmp_path):
    """load(entries) replaces the tuning table; the empty one comes back afterwards."""
    path = str(tmp_path / "tune.json")

    def load(entries):
        text = ",\n".join(f'    "{k}": {v}' for k, v in entries.items())
        open(path, "w").write('{\n  "format": "mfx-autotune-2",\n  "entries": {\n' + text + "\n  }\n}\n")
        assert mfx.load().mfx_autotune_load(path.encode()) == 0

    yield load
    load({})


def chain(h, n, count=4):
    mats = [torch.empty((n, n), device=DEV) for _ in range(count)]
    for i, x in enumerate(mats):
        h.fill_uniform(x, 37, i)
    return mats, [torch.empty((n, n), device=DEV) for _ in range(count - 2)], torch.full((n, n), float("nan"), device=DEV)


def recorded(h, mats, scratch, out, prec):
    h.timing_begin()
    h.chain(mats, scratch, out, prec=prec)
    rec = h.timing_end()
    h.grouped_status()
    want = mats[0].double() @ mats[1].double() @ mats[2].double() @ mats[3].double()
    assert torch.linalg.norm(out.double() - want) < 2 * TOL[prec] * torch.linalg.norm(want)
    return rec


@pytest.mark.parametrize("prec,key", [("fp32", "0:9:9:9"), ("split-bf16", "1:9:9:9"), ("bf16", "2:9:9:9")])
def test_unknown_configuration_in_the_table(handle, mfx, table, prec, key):
    """A product refuses such an id; a list of such products runs as the grouped launch, which does not use it."""
    print(f"unknown configuration {prec}", flush=True)
    mats, scratch, out = chain(handle, 500)
    assert not any(x.startswith("grouped_") for x in recorded(handle, mats, scratch, out, prec))
    table({key: 60})
    out.fill_(float("nan"))
    assert any(x.startswith("grouped_") for x in recorded(handle, mats, scratch, out, prec))
    with pytest.raises(mfx.MfxError) as e:
        handle.gemm(mats[0], mats[1], out, prec=prec)
    assert e.value.status == 1


@pytest.mark.parametrize("prec", ["fp32", "split-bf16", "bf16"])
def test_tuning_keeps_the_dense_form(handle, mfx, table, tmp_path, prec):
    """A list that runs as dense launches by a wide margin still does once it is tuned, also from a saved table."""
    print(f"tuned list {prec}", flush=True)
    mats, scratch, out = chain(handle, 1024)
    pairs = [(mats[0], mats[1], scratch[0]), (mats[2], mats[3], scratch[1]), (scratch[0], scratch[1], out)]
    policy = handle.autotune_grouped([mfx.problem(*p) for p in pairs], [(2, 0), (2, 1)], prec=prec)
    assert 0 <= policy < mfx.grouped_policy_count()
    assert not any(x.startswith("grouped_") for x in recorded(handle, mats, scratch, out, prec))
    path = str(tmp_path / "saved.json").encode()
    assert mfx.load().mfx_autotune_save(path) == 0
    table({})
    assert mfx.load().mfx_autotune_load(path) == 0
    out.fill_(float("nan"))
    assert not any(x.startswith("grouped_") for x in recorded(handle, mats, scratch, out, prec))
    handle.force_grouped_policy(policy)  # a forced policy is still one
    try:
        assert any(x.startswith("grouped_") for x in recorded(handle, mats, scratch, out, prec))
    finally:
        handle.force_grouped_policy(-1)


def test_a_tuned_policy_is_kept(handle, mfx, table):
    """A table's policy still takes the list from the dense form."""
    mats, scratch, out = chain(handle, 1024)
    assert not any(x.startswith("grouped_") for x in recorded(handle, mats, scratch, out, "fp32"))
    # three problems, the square root of their volume in the bucket of 2^16, two levels
    table({"g0:2:16:1": 20})
    assert any(x.startswith("grouped_") for x in recorded(handle, mats, scratch, out, "fp32"))


def test_independent_packed_products_near_the_line(handle, mfx):
    """Estimated at 0.82 of the grouped launch as dense launches, six independent products that are packed run grouped."""
    print("independent packed products", flush=True)
    shapes = [(518, 339, 1151), (163, 1448, 590), (667, 268, 714), (1742, 1815, 678), (501, 176, 2006), (392, 392, 392)]
    ops = []
    for i, (m, n, k) in enumerate(shapes):
        A, B = torch.empty((m, k), device=DEV), torch.empty((k, n), device=DEV)
        handle.fill_uniform(A, 41, 2 * i)
        handle.fill_uniform(B, 41, 2 * i + 1)
        ops.append((A, B, torch.full((m, n), float("nan"), device=DEV)))
    handle.timing_begin()
    handle.grouped([mfx.problem(*o) for o in ops], [], prec="bf16")
    rec = handle.timing_end()
    handle.grouped_status()
    assert any(x.startswith("grouped_") for x in rec)
    for A, B, C in ops:
        want = A.double() @ B.double()
        assert torch.linalg.norm(C.double() - want) < TOL["bf16"] * torch.linalg.norm(want)

"""Short grouped lists that run as dense launches (GPU, through the C ABI):
which lists do, that a grouped launch of the same list agrees, that graph
replays equal the eager call, and that the status calls succeed either way.
Bar: relative Frobenius error against FP64 on U[-1, 1) inputs, 2e-6 (FP32)
or 1e-5 / 1e-2 (split / single BF16) per product on the path."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = {"fp32": 2e-6, "split-bf16": 1e-5, "bf16": 1e-2}


def seeded(h, rows, cols, mid):
    x = torch.empty((rows, cols), device=DEV)
    h.fill_uniform(x, 17, mid)
    return x


def rel(got, want):
    return (torch.linalg.norm(got.double() - want) / torch.linalg.norm(want)).item()


@pytest.mark.parametrize("prec", ["fp32", "split-bf16", "bf16"])
@pytest.mark.parametrize("m,n,k,dense", [(1024, 1024, 1024, True), (1000, 1030, 1026, True), (64, 64, 64, False)])
def test_two_level_list(handle, mfx, prec, m, n, k, dense):
    """Three products, the last of the first two's results, plus an empty and
    a K = 0 problem; the small list stays one grouped launch."""
    print(f"list {prec} {m}x{n}x{k}", flush=True)
    A, B = seeded(handle, m, k, 0), seeded(handle, k, n, 1)
    P, Q = seeded(handle, n, k, 2), seeded(handle, k, m, 3)
    C0 = seeded(handle, m, m, 4)
    E, F, G = (torch.full(s, float("nan"), device=DEV) for s in ((m, n), (n, m), (m, m)))
    Z = seeded(handle, 40, 24, 5)
    Z0 = Z.clone()
    none = torch.empty((0, n), device=DEV)
    def problems():
        return [mfx.problem(A, B, E), mfx.problem(P, Q, F), mfx.problem(E, F, G, alpha=0.5, beta=0.25),
                mfx.problem(torch.empty((0, k), device=DEV), B, none),
                mfx.problem(torch.empty((40, 0), device=DEV), torch.empty((0, 24), device=DEV), Z, beta=0.5)]
    want = 0.5 * (A.double() @ B.double()) @ (P.double() @ Q.double()) + 0.25 * C0.double()

    G.copy_(C0)
    handle.timing_begin()
    handle.grouped(problems(), [(2, 0), (2, 1)], prec=prec)
    rec = handle.timing_end()
    handle.grouped_status()
    assert any(x.startswith("grouped_") for x in rec) == (not dense), rec
    assert rel(G, want) < 2 * TOL[prec]
    assert torch.equal(Z, Z0 * 0.5)
    eager = G.clone()

    g = handle.graph_create(problems(), [(2, 0), (2, 1)], prec=prec)
    for replay in range(3):
        E.fill_(float("nan"))
        G.copy_(C0)
        seeded(handle, 300, 300, 6) @ seeded(handle, 300, 300, 7)  # other work between replays
        g.launch()
        g.status()
        assert torch.equal(G, eager), replay
    g.close()

    handle.force_grouped_policy(3)  # the same list as a grouped launch
    try:
        G.copy_(C0)
        handle.grouped(problems(), [(2, 0), (2, 1)], prec=prec)
        handle.grouped_status()
    finally:
        handle.force_grouped_policy(-1)
    assert rel(G, want) < 2 * TOL[prec]

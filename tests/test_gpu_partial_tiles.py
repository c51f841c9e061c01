"""Where split-K partial tiles live (GPU, through the C ABI): calls of one
handle on several streams at once, calls captured into a caller's graph, on a
fresh handle and with a reserved workspace. Bar: relative Frobenius error
against FP64 on U[-1, 1) inputs, 2e-6 (FP32) or 1e-5 / 1e-2 (split / single BF16)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = {"fp32": 2e-6, "split-bf16": 1e-5, "bf16": 1e-2}


def seeded(h, rows, cols, mid):
    x = torch.empty((rows, cols), device=DEV)
    h.fill_uniform(x, 29, mid)
    return x


def rel(got, want):
    return (torch.linalg.norm(got.double() - want) / torch.linalg.norm(want)).item()


class Call:
    """One product, its FP64 value and a fresh result."""

    def __init__(self, h, kind, prec, m, n, k, mid):
        print(f"partial tiles {kind} {prec} {m}x{n}x{k}", flush=True)
        self.kind, self.prec = kind, prec
        self.A = seeded(h, m, k, mid)
        self.B = seeded(h, k, n, mid + 1) if kind == "gemm" else seeded(h, n, k, mid + 1)
        self.C = torch.empty((m, n), device=DEV)
        A, B = self.A.double(), self.B.double()
        self.want = A @ B if kind == "gemm" else A @ A.T if kind == "syrk" else A @ B.T + B @ A.T

    def run(self, h, stream=None):
        if self.kind == "gemm":
            h.gemm(self.A, self.B, self.C, prec=self.prec, stream=stream)
        elif self.kind == "syrk":
            h.syrk(self.A, self.C, prec=self.prec, stream=stream)
        else:
            h.syr2k(self.A, self.B, self.C, prec=self.prec, stream=stream)

    def recorded(self, h, stream=None):
        h.timing_begin()
        self.run(h, stream)
        return h.timing_end()

    def check(self):
        torch.cuda.synchronize()
        assert rel(self.C, self.want) < TOL[self.prec]


FP32_CALLS = [("syrk", 3000, 3000, 2500), ("syr2k", 4096, 4096, 1024), ("gemm", 3000, 3000, 1500)]


@pytest.mark.parametrize("kind,m,n,k", FP32_CALLS)
def test_two_streams_one_handle(handle, kind, m, n, k):
    calls = [Call(handle, kind, "fp32", m, n, k, 10 * i) for i in (0, 1)]
    streams = [torch.cuda.Stream() for _ in calls]
    alone = []
    for c in calls:
        assert "splitk_reduce" in c.recorded(handle)
        c.check()
        alone.append(c.C.clone())
    torch.cuda.synchronize()
    for _ in range(10):
        for c, s in zip(calls, streams):
            c.run(handle, s)
    torch.cuda.synchronize()
    for c, want in zip(calls, alone):
        assert torch.equal(c.C, want)


def test_more_streams_than_buffers(mfx, handle):
    """The first eight streams of a handle split; further ones run whole tiles."""
    h = mfx.Handle(0)
    c = Call(handle, "syrk", "fp32", 3000, 3000, 2500, 0)
    torch.cuda.synchronize()
    seen = {}
    for i in range(12):
        s = torch.cuda.Stream()
        split = "splitk_reduce" in c.recorded(h, s)
        s.synchronize()
        c.check()
        c.C.fill_(float("nan"))
        torch.cuda.synchronize()
        seen.setdefault(s.cuda_stream, split)
    assert list(seen.values()) == [i < 8 for i in range(len(seen))], seen
    h.close()


def captured(h, c):
    """c.run on h in a graph of its own, replayed with other work between the replays."""
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        c.run(h)
    for _ in range(3):
        c.C.fill_(float("nan"))
        g.replay()
        c.check()
        seeded(h, 300, 300, 6) @ seeded(h, 300, 300, 7)
    return g


@pytest.mark.parametrize("kind,m,n,k", FP32_CALLS)
def test_capture_on_a_fresh_handle(mfx, handle, kind, m, n, k):
    """Holds no library memory, so a later call that regrows the workspace changes nothing."""
    c = Call(handle, kind, "fp32", m, n, k, 0)
    c.run(handle)  # code objects loaded
    h = mfx.Handle(0)
    g = captured(h, c)
    for size in (512, 4096):
        X = seeded(h, size, size, 3)
        h.gemm(X, X, torch.empty((size, size), device=DEV), prec="split-bf16")
        c.run(h)  # eager, on a buffer of the stream
        c.check()
        c.C.fill_(float("nan"))
        g.replay()
        c.check()
    del g
    h.close()


@pytest.mark.parametrize("reserve", [False, True])
def test_capture_of_few_tiles(mfx, handle, reserve):
    """A reserved workspace keeps the k slices of a product on few tiles, bit for bit."""
    m, n, k = 512, 512, 8192
    c = Call(handle, "gemm", "fp32", m, n, k, 0)
    assert "splitk_reduce" in c.recorded(handle)
    eager = c.C.clone()
    h = mfx.Handle(0)
    if reserve:
        h.reserve_workspace(h.lib.mfx_gemm_workspace_size(mfx.FP32, m, n, k))
    g = captured(h, c)
    assert not reserve or torch.equal(c.C, eager)
    del g
    h.close()


@pytest.mark.parametrize("prec,kind,n,k", [("split-bf16", "syr2k", 4096, 1024), ("split-bf16", "syr2k", 3000, 700),
                                           ("split-bf16", "syrk", 3000, 2500), ("bf16", "syr2k", 3000, 2500)])
def test_workspace_of_the_query_is_enough(mfx, handle, prec, kind, n, k):
    """With the workspace that the product query names, the symmetric calls of the same sizes are captured,
    and eager ones take no further memory than their stream's buffer."""
    c = Call(handle, kind, prec, n, n, k, 0)
    assert "splitk_reduce" in c.recorded(handle)
    c.check()
    h = mfx.Handle(0)
    h.reserve_workspace(h.lib.mfx_gemm_workspace_size(mfx.PRECISIONS[prec], n, n, k))
    others = [c, Call(handle, "syrk", prec, n, n, k, 4), Call(handle, "gemm", prec, n, n, k, 8)]
    g = captured(h, c)
    c.run(h)
    for other in others:
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        other.run(h)
        torch.cuda.synchronize()
        assert torch.cuda.mem_get_info()[0] == free, other.kind
        other.check()
    del g
    h.close()


def test_captured_call_outlives_later_eager_calls(mfx, handle):
    """A captured product's packed operands stay where they are while symmetric calls and lists of the same sizes run."""
    n, k = 4096, 1024
    c = Call(handle, "gemm", "split-bf16", n, n, k, 0)
    two = Call(handle, "syr2k", "split-bf16", n, n, k, 4)
    mats = [seeded(handle, 1024, 1024, 10 + i) for i in range(4)]
    scratch, out = [torch.empty((1024, 1024), device=DEV) for _ in range(2)], torch.empty((1024, 1024), device=DEV)
    c.run(handle)
    h = mfx.Handle(0)
    h.reserve_workspace(h.lib.mfx_gemm_workspace_size(mfx.SPLIT_BF16, n, n, k))
    g = captured(h, c)
    for _ in range(3):
        two.run(h)
        two.check()
        h.chain(mats, scratch, out, prec="split-bf16")
        c.C.fill_(float("nan"))
        g.replay()
        c.check()
        assert rel(out, mats[0].double() @ mats[1].double() @ mats[2].double() @ mats[3].double()) < 2 * TOL["split-bf16"]
    del g
    h.close()

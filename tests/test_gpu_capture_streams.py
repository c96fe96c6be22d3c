"""Products with k partitions in captured graphs: captured on a stream that has
made no product before, larger than the stream's eager ones, and replayed beside
eager products and other graphs on other streams. Every result has the bits of
an eager product that had the GPU to itself."""
from __future__ import annotations

import ctypes as C

import pytest
import torch

from tests.conftest import say

pytestmark = pytest.mark.gpu

LOWER = 0xC0


class Product:
    """C := A B with partitions in eager and captured calls alike (m, n <= k/4
    and k >= 2048)."""

    def __init__(self, blis, seed, m, n, k):
        g = torch.Generator(device="cuda").manual_seed(seed)
        self.blis, self.dims = blis, (m, n, k)
        self.a = torch.rand(k, m, generator=g, device="cuda", dtype=torch.float64) - 0.5
        self.b = torch.rand(n, k, generator=g, device="cuda", dtype=torch.float64) - 0.5
        self.out = torch.empty(n, m, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()

    def call(self, out=None):
        m, n, k = self.dims
        one, zero = C.byref(C.c_double(1.0)), C.byref(C.c_double(0.0))
        dst = self.out if out is None else out
        self.blis.bli_dgemm(0, 0, m, n, k, one, self.a.data_ptr(), 1, m, self.b.data_ptr(), 1, k,
                            zero, dst.data_ptr(), 1, m)

    def alone(self, st):
        self.blis.bli_amd_set_stream(st.cuda_stream, 0)
        self.call()
        torch.cuda.synchronize()
        return self.out.clone()

    def capture(self, st):
        self.blis.bli_amd_set_stream(st.cuda_stream, 0)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=st):
            self.call()
        return graph


@pytest.fixture
def own_stream(blis):
    yield
    torch.cuda.synchronize()
    blis.bli_amd_set_stream(None, 1)


def test_capture_on_a_stream_without_products(blis, own_stream):
    say("capture: warmed up on one stream, captured on others")
    warm = torch.cuda.Stream()
    small, large = Product(blis, 1, 128, 96, 8192), Product(blis, 2, 700, 650, 4096)
    want = {p: p.alone(warm) for p in (small, large)}
    fresh = torch.cuda.Stream()
    after_small = torch.cuda.Stream()
    small.alone(after_small)            # its eager buffer is too small for `large`
    for p, st in ((small, fresh), (large, fresh), (large, after_small)):
        graph = p.capture(st)
        for _ in range(3):
            p.out.fill_(7.0)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(p.out, want[p])
            small.alone(warm)


def test_captured_solve_on_a_stream_without_products(blis, own_stream):
    """A solve whose update takes two k partitions by its own rule."""
    say("capture: solve with a partitioned update")
    q, r = 1600, 100
    g = torch.Generator(device="cuda").manual_seed(3)
    a = (torch.rand(q, q, generator=g, device="cuda", dtype=torch.float64) - 0.5) / q ** 0.5
    a.diagonal().add_(1.5)
    b0 = torch.rand(r, q, generator=g, device="cuda", dtype=torch.float64) - 0.5
    x = b0.clone()

    def call():
        blis.bli_dtrsm(0, LOWER, 0, 0, q, r, C.byref(C.c_double(1.0)), a.data_ptr(), 1, q,
                       x.data_ptr(), 1, q)

    torch.cuda.synchronize()
    blis.bli_amd_set_stream(torch.cuda.Stream().cuda_stream, 0)
    call()
    torch.cuda.synchronize()
    want = x.clone()
    st = torch.cuda.Stream()
    blis.bli_amd_set_stream(st.cuda_stream, 0)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        call()
    for _ in range(3):
        x.copy_(b0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(x, want)


def test_graphs_beside_eager_products(blis, own_stream):
    """Two graphs captured on one stream, replayed on two others while that
    stream makes eager products: each has partitions of its own."""
    say("capture: two graphs and eager products side by side")
    reps = 20
    st, r1, r2 = (torch.cuda.Stream() for _ in range(3))
    p1, p2, p3 = (Product(blis, 10 + i, 300, 280, 6000) for i in range(3))
    want = {p: p.alone(st) for p in (p1, p2, p3)}
    g1, g2 = p1.capture(st), p2.capture(st)
    outs = [torch.empty_like(p3.out) for _ in range(reps)]
    blis.bli_amd_set_stream(st.cuda_stream, 0)
    for p in (p1, p2):
        p.out.fill_(7.0)
    torch.cuda.synchronize()
    for i in range(reps):
        with torch.cuda.stream(r1):
            g1.replay()
        with torch.cuda.stream(r2):
            g2.replay()
        p3.call(outs[i])
    torch.cuda.synchronize()
    assert torch.equal(p1.out, want[p1]) and torch.equal(p2.out, want[p2])
    for o in outs:
        assert torch.equal(o, want[p3])


def test_eager_product_grows_its_buffer_beside_a_capture(blis, own_stream):
    """While one stream is captured, a product on another needs more room than
    its stream has: neither disturbs the other."""
    say("capture: an eager product on another stream in its midst")
    st, side = torch.cuda.Stream(), torch.cuda.Stream()
    small, large = Product(blis, 20, 128, 96, 8192), Product(blis, 21, 900, 850, 4096)
    want = {p: p.alone(torch.cuda.Stream()) for p in (small, large)}
    small.alone(side)
    for p in (small, large):
        p.out.fill_(7.0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        blis.bli_amd_set_stream(st.cuda_stream, 0)
        small.call()
        blis.bli_amd_set_stream(side.cuda_stream, 0)
        large.call()
    torch.cuda.synchronize()
    assert torch.equal(large.out, want[large])
    for _ in range(3):
        small.out.fill_(7.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(small.out, want[small])


def test_products_in_flight_on_more_streams_than_buffers(blis, own_stream):
    """A stream beyond the eighth takes the longest unused buffer, whose product
    may still run: nothing is waited for between the calls."""
    say("streams: products in flight on twelve streams")
    p = Product(blis, 22, 600, 550, 6000)
    want = p.alone(torch.cuda.Stream())
    streams = [torch.cuda.Stream() for _ in range(12)]
    outs = [torch.empty_like(want) for _ in range(36)]
    torch.cuda.synchronize()
    for i, o in enumerate(outs):
        blis.bli_amd_set_stream(streams[i % 12].cuda_stream, 0)
        p.call(o)
    torch.cuda.synchronize()
    for o in outs:
        assert torch.equal(o, want)


@pytest.mark.parametrize("rs", [1, 2])
def test_captured_solve_of_a_large_dominant_triangle(blis, own_stream, rs):
    """Captured, it is solved by substitution (inverted blocks need a check that
    the host reads). Bound: as test_gpu_trsm_blocks.py's."""
    q, r = 1600, 520
    say(f"capture: large dominant solve rs={rs}")
    g = torch.Generator(device="cuda").manual_seed(30)
    a = torch.tril(torch.rand(q, q, generator=g, device="cuda", dtype=torch.float64) - 0.5)
    a.diagonal().copy_(torch.rand(q, generator=g, device="cuda", dtype=torch.float64) + q)
    buf = torch.full((q, rs * q), float("nan"), dtype=torch.float64, device="cuda")
    buf[:, ::rs] = a.T
    b0 = torch.rand(r, q, generator=g, device="cuda", dtype=torch.float64) - 0.5
    x = b0.clone()

    def call():
        blis.bli_dtrsm(0, LOWER, 0, 0, q, r, C.byref(C.c_double(1.0)), buf.data_ptr(), rs, rs * q,
                       x.data_ptr(), 1, q)

    def check():
        res = a @ x.T.contiguous() - b0.T
        assert res.norm() <= 8 * q * 2.0 ** -53 * a.norm() * x.norm()

    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    blis.bli_amd_set_stream(st.cuda_stream, 0)
    # Eager first, by inverted blocks and (a row that is not dominant) by
    # substitution, which sizes the workspace that a captured update packs into.
    call()
    torch.cuda.synchronize()
    check()
    off = buf[0, 100 * rs].item()
    buf[0, 100 * rs] = 1e4
    x.copy_(b0)
    torch.cuda.synchronize()
    call()
    torch.cuda.synchronize()
    buf[0, 100 * rs] = off
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        call()
    for _ in range(3):
        x.copy_(b0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        check()

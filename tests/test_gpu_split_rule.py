"""The k partitions that products and masked products (gemmt, syrk) take by
shape (gemm_choose_split, gemm.hip) and the reduction that forms C from them.

* Against FP64 products at shapes around the rule's edges: k at and past 512,
  outputs of one tile, of few and ragged tiles, deep and shallow; both types,
  both triangles, beta zero with NaN in C, non-unit row stride of C.
* Two streams at once: products that take partitions have scratch of their
  own per stream.
* Under stream capture: a product that takes no partitions there replays to
  the bits of one pass.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

from tests.conftest import say, unit_roundoff

pytestmark = pytest.mark.gpu

LOWER, UPPER = 0xC0, 0x60


def _ct(dt):
    return C.c_double if dt == torch.float64 else C.c_float


def _ch(dt):
    return "d" if dt == torch.float64 else "s"


def _u(dt):
    return unit_roundoff(np.float64 if dt == torch.float64 else np.float32)


def _rand(g, dt, *s):
    return torch.rand(*s, generator=g, device="cuda", dtype=dt) * 2 - 1


# (m, n, k): one pass at 512, partitions past it, a k tail in the last
# partition, one 64 x 64 tile, one row of tiles, ragged both ways.
GEMM_SHAPES = [(256, 256, 512), (256, 256, 577), (65, 64, 4099), (64, 64, 3000), (70, 3001, 1500),
               (513, 257, 2049), (1000, 333, 1031), (33, 5, 20000)]


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
@pytest.mark.parametrize("beta", [0.0, -0.5])
def test_gemm_partitions_against_fp64(blis, dt, beta):
    g = torch.Generator(device="cuda").manual_seed(3)
    for m, n, k in GEMM_SHAPES:
        for rs in (1, 2):
            say(f"split rule gemm {dt} beta={beta} {m}x{n}x{k} rs={rs}")
            a, b = _rand(g, dt, m, k), _rand(g, dt, k, n)
            c0 = _rand(g, dt, m, n)
            buf = torch.full((n, m * rs + 3), float("nan"), dtype=dt, device="cuda")
            if beta != 0.0:
                buf[:, :m * rs:rs] = c0.T
            at, bt = a.T.contiguous(), b.T.contiguous()
            getattr(blis, f"bli_{_ch(dt)}gemm")(
                0, 0, m, n, k, C.byref(_ct(dt)(0.75)), at.data_ptr(), 1, m, bt.data_ptr(), 1, k,
                C.byref(_ct(dt)(beta)), buf.data_ptr(), rs, m * rs + 3)
            ref = 0.75 * (a.double() @ b.double()) + beta * c0.double()
            scale = 0.75 * a.double().norm() * b.double().norm() + abs(beta) * c0.double().norm()
            got = buf[:, :m * rs:rs].T.double()
            assert (got - ref).norm() / scale <= 4 * (k + 2) * _u(dt)
            assert torch.isnan(buf[:, m * rs:]).all()
            if rs == 2:
                assert torch.isnan(buf[:, 1:m * rs:2]).all()


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
def test_same_bits_for_c_by_rows_and_by_columns(blis, dt):
    """Shapes far from square, whose best tiles differ in the two orders."""
    g = torch.Generator(device="cuda").manual_seed(8)
    for m, n, k in [(793, 975, 1670), (165, 1931, 6413), (1931, 165, 6413), (4000, 300, 900),
                    (130, 700, 577)]:
        say(f"split rule storage of C {dt} {m}x{n}x{k}")
        a, b = _rand(g, dt, k, m), _rand(g, dt, n, k)
        out = []
        for rows in (False, True):
            c = torch.empty((m, n) if rows else (n, m), dtype=dt, device="cuda")
            getattr(blis, f"bli_{_ch(dt)}gemm")(
                0, 0, m, n, k, C.byref(_ct(dt)(1.0)), a.data_ptr(), 1, m, b.data_ptr(), 1, k,
                C.byref(_ct(dt)(0.0)), c.data_ptr(), n if rows else 1, 1 if rows else m)
            out.append(c if rows else c.T)
        assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
@pytest.mark.parametrize("uplo", [LOWER, UPPER])
@pytest.mark.parametrize("trans", [0, 8])
def test_syrk_partitions_against_fp64(blis, dt, uplo, trans):
    g = torch.Generator(device="cuda").manual_seed(4)
    for n, k in [(1, 700), (63, 512), (65, 577), (130, 4099), (257, 1025), (500, 9001), (33, 40000)]:
        for beta in (0.0, 0.5):
            say(f"split rule syrk {dt} uplo={uplo:x} trans={trans} n={n} k={k} beta={beta}")
            x = _rand(g, dt, n, k)
            st = x.contiguous() if trans else x.T.contiguous()   # column-major op storage
            c0 = _rand(g, dt, n, n)
            c = c0.T.clone(memory_format=torch.contiguous_format)
            if beta == 0.0:
                c.fill_(float("nan"))
            getattr(blis, f"bli_{_ch(dt)}syrk")(
                uplo, trans, n, k, C.byref(_ct(dt)(-1.5)), st.data_ptr(), 1, k if trans else n,
                C.byref(_ct(dt)(beta)), c.data_ptr(), 1, n)
            keep = torch.tril(torch.ones(n, n, dtype=torch.bool, device="cuda"))
            keep = keep if uplo == LOWER else keep.T
            xd = x.double()
            ref = -1.5 * (xd @ xd.T.contiguous()) + beta * c0.double()
            got = c.T
            scale = 1.5 * xd.norm() ** 2 + beta * c0.double().norm()
            assert (got[keep].double() - ref[keep]).norm() / scale <= 4 * (k + 2) * _u(dt)
            rest = got[~keep]
            assert torch.isnan(rest).all() if beta == 0.0 else torch.equal(rest, c0[~keep])


def _calls(blis, st, ops, reps):
    """reps x C := A B on stream st, asynchronous, into fresh outputs."""
    one, zero = C.byref(C.c_double(1.0)), C.byref(C.c_double(0.0))
    a, b, m, n, k = ops
    outs = [torch.empty(n, m, dtype=torch.float64, device="cuda") for _ in range(reps)]
    torch.cuda.synchronize()
    blis.bli_amd_set_stream(st.cuda_stream, 0)
    return outs, lambda i: (blis.bli_amd_set_stream(st.cuda_stream, 0),
                            blis.bli_dgemm(0, 0, m, n, k, one, a.data_ptr(), 1, m, b.data_ptr(),
                                           1, k, zero, outs[i].data_ptr(), 1, m))


def test_two_streams_do_not_share_partitions(blis):
    say("split rule: two streams interleaved")
    g = torch.Generator(device="cuda").manual_seed(5)
    m, n, k, reps = 300, 280, 6000, 20
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    ops = [( _rand(g, torch.float64, k, m), _rand(g, torch.float64, n, k), m, n, k)
           for _ in range(2)]
    try:
        o1, f1 = _calls(blis, s1, ops[0], reps)
        o2, f2 = _calls(blis, s2, ops[1], reps)
        for i in range(reps):
            f1(i)
            f2(i)
        torch.cuda.synchronize()
        for outs in (o1, o2):
            for o in outs[1:]:
                assert torch.equal(o, outs[0])
        # The first of each against a call that had the GPU to itself.
        for ops_, outs, st in ((ops[0], o1, s1), (ops[1], o2, s2)):
            alone, f = _calls(blis, st, ops_, 1)
            f(0)
            torch.cuda.synchronize()
            assert torch.equal(alone[0], outs[0])
    finally:
        blis.bli_amd_set_stream(None, 1)


def test_captured_product_takes_one_pass(blis):
    say("split rule: captured product")
    g = torch.Generator(device="cuda").manual_seed(6)
    m, n, k = 500, 400, 1200        # partitions in an eager call, one pass when captured
    a, b = _rand(g, torch.float64, k, m), _rand(g, torch.float64, n, k)
    out = torch.empty(n, m, dtype=torch.float64, device="cuda")
    one, zero = C.byref(C.c_double(1.0)), C.byref(C.c_double(0.0))

    def call():
        blis.bli_dgemm(0, 0, m, n, k, one, a.data_ptr(), 1, m, b.data_ptr(), 1, k, zero,
                       out.data_ptr(), 1, m)

    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    try:
        blis.bli_amd_set_stream(st.cuda_stream, 0)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=st):
            call()
        blis.bli_amd_gemm_set_config(3, 8, 1, 1)
        call()
        torch.cuda.synchronize()
        want = out.clone()
        blis.bli_amd_gemm_set_config(-1, 8, 1, 1)
        for _ in range(3):
            out.fill_(7.0)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
    finally:
        blis.bli_amd_gemm_set_config(-1, 8, 1, 1)
        blis.bli_amd_set_stream(None, 1)


def test_partitions_in_a_graph_outlive_other_streams(blis):
    """A graph holds the address of its stream's partitions: the first products
    of more streams than the library keeps buffers for, and a larger product on
    the same stream, leave them alone."""
    say("split rule: partitions held by a graph")
    g = torch.Generator(device="cuda").manual_seed(7)
    m, n, k = 128, 96, 8192          # split under capture too
    a, b = _rand(g, torch.float64, k, m), _rand(g, torch.float64, n, k)
    out, other = (torch.empty(n, m, dtype=torch.float64, device="cuda") for _ in range(2))
    big_a, big_b = _rand(g, torch.float64, 4096, 700), _rand(g, torch.float64, 700, 4096)
    big = torch.empty(700, 700, dtype=torch.float64, device="cuda")
    one, zero = C.byref(C.c_double(1.0)), C.byref(C.c_double(0.0))

    def call(dst):
        blis.bli_dgemm(0, 0, m, n, k, one, a.data_ptr(), 1, m, b.data_ptr(), 1, k, zero,
                       dst.data_ptr(), 1, m)

    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    try:
        blis.bli_amd_set_stream(st.cuda_stream, 0)
        call(out)
        torch.cuda.synchronize()
        want = out.clone()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=st):
            call(out)
        for _ in range(3):
            for s in [torch.cuda.Stream() for _ in range(9)]:
                blis.bli_amd_set_stream(s.cuda_stream, 0)
                other.fill_(7.0)
                torch.cuda.synchronize()
                call(other)
                torch.cuda.synchronize()
                assert torch.equal(other, want)
            blis.bli_amd_set_stream(st.cuda_stream, 0)
            blis.bli_dgemm(0, 0, 700, 700, 4096, one, big_a.data_ptr(), 1, 700, big_b.data_ptr(),
                           1, 4096, zero, big.data_ptr(), 1, 700)
            out.fill_(7.0)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
    finally:
        blis.bli_amd_set_stream(None, 1)

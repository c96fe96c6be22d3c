"""How the GEMM tiles read their operands (SlabLoader, gemm_tile.hpp).

Every tile reads A and B through buffer descriptors that end at the operand's
last element; operands whose strides do not allow that (negative, overlapping
or very large leading dimensions) take the loads behind bounds checks. The
arithmetic is the same either way, so a product of the same values with the
same k partition (one pass on a given tile, or the default path's) must have
the same bits whatever the storage: leading dimensions of every residue, a
base that is aligned to one element only, memory full of NaN between and
around the columns, reversed columns.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

from tests.conftest import say, unit_roundoff

pytestmark = pytest.mark.gpu

# Tile edges: below, at and above the 16/32/64/128 tiles and the 8 to 64 deep
# k slabs, with remainders of every 16-byte vector.
SHAPES = [(1, 3, 1), (31, 33, 15), (64, 65, 17), (129, 127, 66), (200, 131, 513), (515, 258, 33)]


def _store(x, pad, off, reverse=False):
    """x (rows x cols) column-major in a NaN-filled device buffer with `pad`
    extra rows between columns, starting `off` elements in; reversed: the
    columns run backwards. Returns (buffer, address of (0, 0), cs)."""
    r, c = x.shape
    ld = r + pad
    buf = torch.full((off + ld * c + off,), float("nan"), dtype=x.dtype, device="cuda")
    v = buf[off:off + ld * c].view(c, ld)
    v[:, :r] = (x.flip(1) if reverse else x).T
    start = buf.data_ptr() + (off + (ld * (c - 1) if reverse else 0)) * x.element_size()
    return buf, start, -ld if reverse else ld


def _run(blis, dt, ta, tb, m, n, k, a, b, c0, pad, off, reverse, tile):
    ch, ct = ("d", C.c_double) if dt == torch.float64 else ("s", C.c_float)
    ba, pa, la = _store(a.T if ta else a, pad, off, reverse)
    bb, pb, lb = _store(b.T if tb else b, pad, off, reverse)
    bc, pc, lc = _store(c0, pad, off)
    if tile is not None:
        blis.bli_amd_gemm_set_config(tile, 8, 1, 1)
    try:
        getattr(blis, f"bli_{ch}gemm")(8 if ta else 0, 8 if tb else 0, m, n, k,
                                       C.byref(ct(1.25)), pa, 1, la, pb, 1, lb,
                                       C.byref(ct(0.5)), pc, 1, lc)
    finally:
        if tile is not None:
            blis.bli_amd_gemm_set_config(-1, 8, 1, 1)
    v = bc[off:off + lc * n].view(n, lc)
    assert torch.isnan(v[:, m:]).all() and torch.isnan(bc[:off]).all() and \
        torch.isnan(bc[off + lc * n:]).all(), "wrote outside C"
    return v[:, :m].T.cpu()


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("tb", [0, 1])
def test_same_bits_for_every_storage(blis, dt, ta, tb):
    g = torch.Generator(device="cuda").manual_seed(ta + 2 * tb)
    u = unit_roundoff(np.float64 if dt == torch.float64 else np.float32)
    tiles = [None, 4, 6 if dt == torch.float64 else 12]
    for m, n, k in SHAPES:
        a, b, c0 = (torch.rand(r, c, generator=g, device="cuda", dtype=dt) * 2 - 1
                    for r, c in ((m, k), (k, n), (m, n)))
        ref = 1.25 * (a.double() @ b.double()) + 0.5 * c0.double()
        scale = 1.25 * a.double().norm() * b.double().norm() + 0.5 * c0.double().norm()
        bases = {}
        for tile in tiles:
            for pad, off, reverse in ((0, 0, False), (1, 1, False), (3, 3, False), (8, 2, False),
                                      (2, 1, True)):
                say(f"loads {dt} ta={ta} tb={tb} {m}x{n}x{k} tile={tile} pad={pad} off={off} "
                    f"reverse={reverse}")
                got = _run(blis, dt, ta, tb, m, n, k, a, b, c0, pad, off, reverse, tile)
                base = bases.setdefault(tile is None, got)
                if base is got:
                    err = (got.cuda().double() - ref).norm() / scale
                    assert err <= 4 * (k + 2) * u
                assert torch.equal(got, base)


def test_leading_dimension_beyond_32_bit_offsets(blis):
    """Columns 2^27 + 1 doubles apart: 32 lines of a slab span more than 4 GiB,
    past what a descriptor's offsets reach, and every column start is odd."""
    m, n, k, ld = 33, 40, 5, (1 << 27) + 1
    say("loads: leading dimension beyond 32-bit offsets")
    g = torch.Generator(device="cuda").manual_seed(7)
    a = torch.rand(m, k, generator=g, device="cuda", dtype=torch.float64)
    b = torch.rand(k, n, generator=g, device="cuda", dtype=torch.float64)
    big = torch.empty(ld * (k - 1) + m, dtype=torch.float64, device="cuda")
    for j in range(k):
        big[j * ld:j * ld + m] = a[:, j]
    tight = a.T.contiguous()
    bt = b.T.contiguous()
    out = []
    for ptr, lda in ((tight.data_ptr(), m), (big.data_ptr(), ld)):
        c = torch.zeros(n, m, dtype=torch.float64, device="cuda")
        blis.bli_dgemm(0, 0, m, n, k, C.byref(C.c_double(1.0)), ptr, 1, lda, bt.data_ptr(), 1, k,
                       C.byref(C.c_double(0.0)), c.data_ptr(), 1, m)
        out.append(c)
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
def test_vectors_with_any_stride_between_lines(blis, dt):
    """An operand of one line (k = 1, m = 1 or n = 1) has no second line: the
    bits do not depend on the stride given for it."""
    g = torch.Generator(device="cuda").manual_seed(21)
    ch, ct = ("d", C.c_double) if dt == torch.float64 else ("s", C.c_float)
    for m, n, k in [(130, 70, 1), (1, 70, 300), (130, 1, 300), (1, 1, 700), (33, 1, 513)]:
        a, b, c0 = (torch.rand(r, c, generator=g, device="cuda", dtype=dt) * 2 - 1
                    for r, c in ((m, k), (k, n), (m, n)))
        base = None
        for ta, tb in ((0, 0), (1, 0), (0, 1), (1, 1)):
            for ld in (None, 1, 0, -3, 1 << 33):
                st, args = [], []
                for x, t, in ((a, ta), (b, tb)):
                    x = (x.T if t else x)
                    buf = x.T.contiguous()               # column-major
                    st.append(buf)
                    args.append(ld if ld is not None and x.shape[1] == 1 else x.shape[0])
                c = c0.T.contiguous()
                say(f"loads one line {dt} {m}x{n}x{k} ta={ta} tb={tb} ld={ld} {args}")
                getattr(blis, f"bli_{ch}gemm")(8 * ta, 8 * tb, m, n, k, C.byref(ct(1.25)),
                                               st[0].data_ptr(), 1, args[0], st[1].data_ptr(), 1,
                                               args[1], C.byref(ct(0.5)), c.data_ptr(), 1, m)
                base = c if base is None else base
                assert torch.equal(c, base)


def _frames(x, hop, rows, length):
    return torch.stack([x[i * hop:i * hop + length] for i in range(rows)])


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
def test_overlapping_frames(blis, dt):
    """Rows of A (or columns of B) that are windows of one signal, a hop apart:
    the bits of the same values stored without overlap."""
    g = torch.Generator(device="cuda").manual_seed(22)
    ch, ct = ("d", C.c_double) if dt == torch.float64 else ("s", C.c_float)
    for rows, cols, k, hop in [(200, 33, 131, 7), (65, 129, 600, 1), (40, 40, 17, 16),
                               (300, 150, 1000, 0), (129, 64, 515, 257)]:
        sig = torch.full((hop * (rows - 1) + k + 64,), float("nan"), dtype=dt, device="cuda")
        sig[:hop * (rows - 1) + k] = torch.rand(hop * (rows - 1) + k, generator=g, device="cuda",
                                                dtype=dt) * 2 - 1
        y = torch.rand(cols, k, generator=g, device="cuda", dtype=dt) * 2 - 1
        tight = _frames(sig, hop, rows, k).contiguous()
        for side in "ab":
            out = []
            for ptr, ld in ((tight.data_ptr(), k), (sig.data_ptr(), hop)):
                say(f"loads frames {dt} {side} {rows}x{cols}x{k} hop={hop} ld={ld}")
                m, n = (rows, cols) if side == "a" else (cols, rows)
                c = torch.zeros(n, m, dtype=dt, device="cuda")
                fa, fb = (ptr, y.data_ptr()) if side == "a" else (y.data_ptr(), ptr)
                la, lb = (ld, k) if side == "a" else (k, ld)
                getattr(blis, f"bli_{ch}gemm")(8, 0, m, n, k, C.byref(ct(1.0)), fa, 1, la, fb, 1,
                                               lb, C.byref(ct(0.0)), c.data_ptr(), 1, m)
                out.append(c)
            assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
def test_batch_plan_takes_vectors_and_frames(blis, dt):
    """A plan runs them in its own kernels (they have work items), with the bits
    of single calls."""
    # (m, n, k, ta, tb, lda, ldb)
    _plan_against_calls(blis, dt, [
        (100, 80, 1, 0, 0, 1, 1), (90, 1, 60, 0, 0, 90, 1), (1, 75, 64, 1, 0, 3, 64),
        (70, 40, 100, 1, 0, 5, 100), (50, 66, 130, 0, 0, 50, 2), (130, 20, 33, 1, 0, 0, 33)])


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
def test_batch_plan_takes_backward_and_overlapping_lines(blis, dt):
    """Strides that descriptors do not take, in either operand and layout, beside
    problems that have none, in every mode of the plan and replayed from its
    graph."""
    _plan_against_calls(blis, dt, [
        (100, 80, 70, 0, 0, -100, 70), (31, 33, 129, 1, 0, -129, 129), (65, 64, 1, 0, 1, 65, -64),
        (64, 1, 300, 1, 0, -300, 300), (33, 97, 40, 0, 0, 33, -41), (17, 15, 16, 0, 0, 5, 16),
        (128, 40, 65, 1, 1, -65, -40), (50, 50, 50, 0, 0, 50, 50), (200, 90, 33, 1, 0, 33, 33)],
        modes=(0, 3, 4, 5, 7, 8))


def _plan_against_calls(blis, dt, probs, modes=(None,)):
    ch, ct = ("d", C.c_double) if dt == torch.float64 else ("s", C.c_float)
    g = torch.Generator(device="cuda").manual_seed(23)
    # (0, 0) of both operands lies in the middle of the buffer: lines may run
    # backwards from there.
    buf = torch.rand(1 << 17, generator=g, device="cuda", dtype=dt) * 2 - 1
    pa, pb = buf[1 << 16:].data_ptr(), buf[(1 << 16) + 1000:].data_ptr()
    one, half = ct(1.0), ct(0.5)
    outs, wants, starts = [], [], []
    for m, n, k, ta, tb, lda, ldb in probs:
        c = torch.rand(n, m, generator=g, device="cuda", dtype=dt)
        w = c.clone()
        getattr(blis, f"bli_{ch}gemm")(8 * ta, 8 * tb, m, n, k, C.byref(one), pa, 1, lda, pb, 1,
                                       ldb, C.byref(half), w.data_ptr(), 1, m)
        outs.append(c)
        starts.append(c.clone())
        wants.append(w)
    real = np.float64 if dt == torch.float64 else np.float32
    col = lambda i, t=np.int64: np.array([p[i] for p in probs], t)
    ones, cnt = np.ones(len(probs), np.int64), len(probs)
    arrs = [col(3, np.int32) * 8, col(4, np.int32) * 8, col(0), col(1), col(2),
            np.full(cnt, 1.0, real), np.full(cnt, pa, np.int64), ones, col(5),
            np.full(cnt, pb, np.int64), ones, col(6), np.full(cnt, 0.5, real),
            np.array([c.data_ptr() for c in outs], np.int64), ones, col(0)]
    arrs = [np.ascontiguousarray(x, x.dtype) for x in arrs]
    torch.cuda.synchronize()
    say(f"loads batch plan {dt}")
    plan = getattr(blis, f"bli_amd_{ch}gemm_batch_plan_create")(
        *[x.ctypes.data for x in arrs], cnt, ones.ctypes.data)
    try:
        assert blis.bli_amd_gemm_batch_plan_work_items(plan) >= cnt
        for mode in modes:
            if mode is not None:
                blis.bli_amd_gemm_batch_plan_set_mode(plan, mode)
            for graph in (0, 1, 1):
                say(f"loads batch plan {dt} mode={mode} graph={graph}")
                for c, c0 in zip(outs, starts):
                    c.copy_(c0)
                torch.cuda.synchronize()
                blis.bli_amd_gemm_batch_plan_execute(plan, graph)
                torch.cuda.synchronize()
                for c, w in zip(outs, wants):
                    assert torch.equal(c, w)
    finally:
        blis.bli_amd_gemm_batch_plan_destroy(plan)

"""Triangular solves whose 512-row diagonal blocks are solved by products with
their inverses (trsm.hip): at least 1536 rows over at least 512 right-hand sides,
every 256-row block of the triangle's diagonal dominant.

Both types, sides, triangles, transposes and diagonals, whole blocks and a
ragged end (solved by substitution), alpha other than 1, right-hand sides padded
and stored by rows, triangles with a unit stride and without, and the way back to
substitution when one block is not dominant. NaN stands in everything that must
not be read.

Bound: ||op(A) X - alpha B||_F <= 8 q u ||A||_F ||X||_F. The diagonal lies in
[1, 2] and the rest of a block's row sums to at most 0.4, so a block's condition
number is at most 3 x 2; the product with its inverse costs at most six times
substitution's 512 u, and the updates q u: 6 x 512 + q < 8 q.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

from tests.conftest import say, unit_roundoff

pytestmark = pytest.mark.gpu

LOWER, UPPER = 0xC0, 0x60


def _triangle(g, dt, q, uplo, unit, one_block_not_dominant):
    """(dense logical triangle, the same with NaN in what is not stored)."""
    a = (torch.rand(q, q, generator=g, device="cuda", dtype=dt) * 2 - 1) / q ** 0.5
    block = torch.arange(q, device="cuda") // 256
    within = block[:, None] == block[None, :]
    if one_block_not_dominant:
        within &= (block != 3)[:, None]
    a = torch.where(within, a * (0.4 * q ** 0.5 / 256), a)
    d = torch.rand(q, generator=g, device="cuda", dtype=dt) + 1
    a.diagonal().copy_(d)
    keep = torch.tril(torch.ones(q, q, dtype=torch.bool, device="cuda"))
    keep = keep if uplo == LOWER else keep.T
    stored = torch.where(keep, a, torch.full_like(a, float("nan")))
    full = torch.where(keep, a, torch.zeros_like(a))
    if unit:
        stored.diagonal().fill_(float("nan"))
        full.diagonal().fill_(1.0)
    return full, stored


def _store(x, rs, cs, fill):
    """x in a buffer of its own with element strides rs, cs."""
    r, c = x.shape
    buf = torch.full(((r - 1) * rs + (c - 1) * cs + 1,), fill, dtype=x.dtype, device="cuda")
    v = buf.as_strided((r, c), (rs, cs))
    v.copy_(x)
    return buf, v


def _check(blis, dt, left, uplo, trans, unit, q, r, alpha=1.0, tri_gap=0, rows_stored=False,
           pad=0, not_dominant=False, seed=31):
    g = torch.Generator(device="cuda").manual_seed(seed)
    ch, ct = ("d", C.c_double) if dt == torch.float64 else ("s", C.c_float)
    u = unit_roundoff(np.float64 if dt == torch.float64 else np.float32)
    full, stored = _triangle(g, dt, q, uplo, unit, not_dominant)
    m, n = (q, r) if left else (r, q)
    b = torch.rand(m, n, generator=g, device="cuda", dtype=dt) * 2 - 1
    nan = float("nan")
    ars, acs = {0: (1, q + pad), 1: (2, 2 * q + 1), 2: (2 * q + 1, 2)}[tri_gap]
    abuf, _ = _store(stored, ars, acs, nan)
    brs, bcs = (n + pad, 1) if rows_stored else (1, m + pad)
    bbuf, x = _store(b, brs, bcs, nan)
    torch.cuda.synchronize()
    say(f"trsm blocks {dt} left={left} uplo={uplo:x} trans={trans} unit={unit} q={q} r={r} "
        f"alpha={alpha} strides={ars},{acs} rows_stored={rows_stored} not_dominant={not_dominant}")
    getattr(blis, f"bli_{ch}trsm")(0 if left else 1, uplo, 8 if trans else 0,
                                   0x100 if unit else 0, m, n, C.byref(ct(alpha)),
                                   abuf.data_ptr(), ars, acs, bbuf.data_ptr(), brs, bcs)
    blis.bli_amd_synchronize()
    op = (full.T if trans else full).double().contiguous()
    xd = x.double().contiguous()
    res = (op @ xd if left else xd @ op) - alpha * b.double()
    assert res.norm() <= 8 * q * u * op.norm() * xd.norm()
    assert int(torch.isnan(bbuf).sum()) == bbuf.numel() - m * n   # the gaps, and they alone


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
@pytest.mark.parametrize("left", [True, False])
@pytest.mark.parametrize("uplo", [LOWER, UPPER])
@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("unit", [False, True])
def test_blocks_by_product(blis, dt, left, uplo, trans, unit):
    _check(blis, dt, left, uplo, trans, unit, 1536, 512)
    _check(blis, dt, left, uplo, trans, unit, 1600, 530, alpha=-0.75, pad=3, rows_stored=left)
    _check(blis, dt, left, uplo, trans, unit, 2100, 515, alpha=2.0, pad=1, not_dominant=True)


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
@pytest.mark.parametrize("uplo", [LOWER, UPPER])
@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("tri_gap", [1, 2])
def test_triangle_without_unit_stride(blis, dt, uplo, trans, tri_gap):
    _check(blis, dt, True, uplo, trans, False, 1700, 520, alpha=0.5, tri_gap=tri_gap)
    _check(blis, dt, False, uplo, trans, True, 1536, 513, tri_gap=tri_gap, rows_stored=True)
    _check(blis, dt, True, uplo, trans, False, 1600, 512, tri_gap=tri_gap, not_dominant=True)


def test_blocks_by_product_asynchronous(blis):
    """Calls that return before the device is done (the solve itself waits once,
    for the check of the diagonal blocks)."""
    blis.bli_amd_set_stream(None, 0)
    try:
        for not_dominant in (False, True):
            _check(blis, torch.float64, True, LOWER, False, False, 1600, 530,
                   not_dominant=not_dominant)
    finally:
        blis.bli_amd_set_stream(None, 1)

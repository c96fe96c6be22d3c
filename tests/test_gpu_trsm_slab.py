"""Triangular solves by substitution (trsm_slab_kernel, trsm.hip).

* Every side, triangle, transpose and diagonal, at row counts around its
  tiles (16 rows, 256 and 512 per launch, recursion beyond) and column counts
  around its 16 columns, with odd leading dimensions, one-element alignment,
  row-stored B, and NaN in everything that must not be read: the residual
  ||op(A) X - alpha B||_F against 2 (q + 2) u ||A||_F ||X||_F, the bound of
  substitution with reciprocal diagonals (gamma_q per element, rounded up).
* An Inf in the right-hand side reaches the rows solved after its own and no
  other row or column.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

from tests.conftest import say, unit_roundoff

pytestmark = pytest.mark.gpu

LOWER, UPPER = 0xC0, 0x60


def _solve(blis, dt, left, uplo, trans, unit, a, b, alpha, pad, rowmajor):
    """X for op(A) X = alpha B (left) or X op(A) = alpha B; a and b dense
    logical matrices, a's unstored part NaN."""
    ch, ct = ("d", C.c_double) if dt == torch.float64 else ("s", C.c_float)
    q = a.shape[0]
    m, n = b.shape
    ab = torch.full((q * (q + pad) + 1,), float("nan"), dtype=dt, device="cuda")
    av = ab[1:].view(q, q + pad)
    av[:, :q] = a.T
    src = b if rowmajor else b.T
    bb = torch.full((src.shape[0] * (src.shape[1] + pad) + 1,), float("nan"), dtype=dt,
                    device="cuda")
    bv = bb[1:].view(src.shape[0], src.shape[1] + pad)
    bv[:, :src.shape[1]] = src
    rs, cs = (bv.shape[1], 1) if rowmajor else (1, bv.shape[1])
    getattr(blis, f"bli_{ch}trsm")(0 if left else 1, uplo, 8 if trans else 0,
                                   0x100 if unit else 0, m, n, C.byref(ct(alpha)),
                                   av.data_ptr(), 1, q + pad, bv.data_ptr(), rs, cs)
    assert torch.isnan(bv[:, src.shape[1]:]).all() and torch.isnan(bb[0])
    x = bv[:, :src.shape[1]]
    return (x if rowmajor else x.T).clone()


def _triangle(g, dt, q, uplo, unit):
    a = (torch.rand(q, q, generator=g, device="cuda", dtype=dt) * 2 - 1) / max(q, 1) ** 0.5
    a.diagonal().copy_(torch.rand(q, generator=g, device="cuda", dtype=dt) + 1)
    full = torch.tril(a) if uplo == LOWER else torch.triu(a)
    stored = torch.where(torch.tril(torch.ones_like(a)).bool() if uplo == LOWER
                         else torch.triu(torch.ones_like(a)).bool(), a,
                         torch.full_like(a, float("nan")))
    if unit:
        stored.diagonal().fill_(float("nan"))
        full.diagonal().fill_(1.0)
    return full, stored


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
@pytest.mark.parametrize("left", [True, False])
@pytest.mark.parametrize("uplo", [LOWER, UPPER])
@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("unit", [False, True])
def test_substitution_residual(blis, dt, left, uplo, trans, unit):
    g = torch.Generator(device="cuda").manual_seed(11)
    u = unit_roundoff(np.float64 if dt == torch.float64 else np.float32)
    for q, r in [(1, 1), (3, 17), (15, 16), (16, 5), (17, 33), (129, 15), (255, 40), (257, 64),
                 (511, 31), (512, 16), (513, 100), (1031, 70)]:
        for pad, rowmajor in ((0, False), (3, True)):
            say(f"trsm slab {dt} left={left} uplo={uplo:x} trans={trans} unit={unit} q={q} r={r} "
                f"pad={pad} rowmajor={rowmajor}")
            full, stored = _triangle(g, dt, q, uplo, unit)
            b = torch.rand(*((q, r) if left else (r, q)), generator=g, device="cuda",
                           dtype=dt) * 2 - 1
            x = _solve(blis, dt, left, uplo, trans, unit, stored, b, -0.75, pad, rowmajor)
            op = (full.T if trans else full).double().contiguous()
            xd = x.double().contiguous()
            res = (op @ xd if left else xd @ op) + 0.75 * b.double()
            assert res.norm() <= 2 * (q + 2) * u * op.norm() * xd.norm()


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
@pytest.mark.parametrize("uplo", [LOWER, UPPER])
def test_infinite_right_hand_side_stays_in_its_rows(blis, dt, uplo):
    g = torch.Generator(device="cuda").manual_seed(12)
    q, r = 300, 20
    full, stored = _triangle(g, dt, q, uplo, False)
    b = torch.rand(q, r, generator=g, device="cuda", dtype=dt) * 2 - 1
    say(f"trsm slab Inf {dt} uplo={uplo:x}")
    clean = _solve(blis, dt, True, uplo, False, False, stored, b, 1.0, 1, False)
    for i in (0, 1, 2, 3, 4, 7, 13, 15, 16, 18, 130, 255, 256, 299):
        bad = b.clone()
        bad[i, 3] = float("inf")
        x = _solve(blis, dt, True, uplo, False, False, stored, bad, 1.0, 1, False)
        before = slice(0, i) if uplo == LOWER else slice(i + 1, q)
        assert torch.equal(x[before, 3], clean[before, 3]), i
        assert torch.isinf(x[i, 3])
        others = [c for c in range(r) if c != 3]
        assert torch.equal(x[:, others], clean[:, others]), i

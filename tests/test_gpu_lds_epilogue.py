"""C written through LDS by the tiles whose lanes hold no whole 16-byte
vectors of it (store_tile_lds, gemm_tile.hpp).

The arithmetic per element is that of the vector epilogue, so every tile of
the table has the bits of the 32 x 32 one, which writes from the
accumulators, at sizes around the tile edges and for every storage of C:
padded columns of odd length, a base aligned to one element, neither stride
one, and beta == 0 over NaN.
"""
from __future__ import annotations

import ctypes as C

import pytest
import torch

from tests.conftest import say

pytestmark = pytest.mark.gpu


def _c(c0, rs, pad, off):
    """c0 (m x n) in a device buffer of -7s, row stride rs, columns m*rs + pad
    apart, `off` elements in. Returns (buffer, the matrix's own view, cs)."""
    m, n = c0.shape
    cs = m * rs + pad
    buf = torch.full((2 * off + cs * n + 4,), -7.0, dtype=c0.dtype, device="cuda")
    v = torch.as_strided(buf, (m, n), (rs, cs), off)
    v.copy_(c0)
    return buf, v, cs


@pytest.mark.parametrize("dt,ch", [(torch.float32, "s"), (torch.float64, "d")])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (3, 130, 5), (63, 65, 33), (128, 128, 64),
                                   (129, 127, 40), (257, 66, 31)])
def test_every_tile_writes_the_same_c(blis, dt, ch, m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, b, c0 = (torch.rand(c, r, generator=g, device="cuda", dtype=dt) * 2 - 1
                for r, c in ((m, k), (k, n), (m, n)))
    ct = C.c_float if ch == "s" else C.c_double
    for rs, pad, off in ((1, 0, 0), (1, 3, 1), (2, 5, 3)):
        for beta in (0.5, 0.0):
            base = None
            for tile in [4] + [t for t in range(14) if t != 4]:
                say(f"lds epilogue {ch} {m}x{n}x{k} rs={rs} pad={pad} beta={beta} tile={tile}")
                start = c0.T if beta else torch.full((m, n), float("nan"), dtype=dt, device="cuda")
                buf, v, cs = _c(start, rs, pad, off)
                outside = buf.clone()
                blis.bli_amd_gemm_set_config(tile, 8, 1, 1)
                try:
                    getattr(blis, f"bli_{ch}gemm")(
                        0, 0, m, n, k, C.byref(ct(1.25)), a.data_ptr(), 1, m, b.data_ptr(), 1, k,
                        C.byref(ct(beta)), v.data_ptr(), rs, cs)
                finally:
                    blis.bli_amd_gemm_set_config(-1, 8, 1, 1)
                got = v.clone()
                assert not torch.isnan(got).any()
                torch.as_strided(outside, (m, n), (rs, cs), off).copy_(got)
                assert torch.equal(buf, outside), "wrote outside C"
                if base is None:
                    base = got
                assert torch.equal(got, base)

"""Captured products past the memory that graphs may hold for k partitions
(1 GiB) are made in one pass. The last file: what graphs hold stays allocated
until the process ends, so captures after it make one pass too."""
from __future__ import annotations

import ctypes as C

import pytest
import torch

from tests.conftest import say

pytestmark = pytest.mark.gpu


def test_captures_past_the_limit_make_one_pass(blis):
    m, n, k = 700, 650, 4096            # about 28 MiB of partitions
    g = torch.Generator(device="cuda").manual_seed(41)
    a = torch.rand(k, m, generator=g, device="cuda", dtype=torch.float64) - 0.5
    b = torch.rand(n, k, generator=g, device="cuda", dtype=torch.float64) - 0.5
    out = torch.empty(n, m, dtype=torch.float64, device="cuda")
    one, zero = C.byref(C.c_double(1.0)), C.byref(C.c_double(0.0))

    def call():
        blis.bli_dgemm(0, 0, m, n, k, one, a.data_ptr(), 1, m, b.data_ptr(), 1, k, zero,
                       out.data_ptr(), 1, m)

    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    try:
        blis.bli_amd_set_stream(st.cuda_stream, 0)
        call()
        torch.cuda.synchronize()
        eager = out.clone()
        blis.bli_amd_gemm_set_config(3, 8, 1, 1)
        call()
        torch.cuda.synchronize()
        single = out.clone()
        blis.bli_amd_gemm_set_config(-1, 8, 1, 1)
        assert not torch.equal(eager, single)       # the partitions round differently
        graphs = []
        for i in range(48):
            say(f"partition limit: capture {i}")
            graphs.append(torch.cuda.CUDAGraph())
            with torch.cuda.graph(graphs[-1], stream=st):
                call()
        for graph, want in ((graphs[0], eager), (graphs[-1], single), (graphs[1], eager)):
            out.fill_(7.0)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
        # Eager products have partitions of their own.
        call()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
    finally:
        torch.cuda.synchronize()
        blis.bli_amd_gemm_set_config(-1, 8, 1, 1)
        blis.bli_amd_set_stream(None, 1)

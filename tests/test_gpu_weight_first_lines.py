"""Outputs on both sides of the lines of ``_weight_first`` for 1025 to 2048 columns: the
launch taken gives the bits of the codes' GEMM."""

from __future__ import annotations

import pytest
import torch

from helpers import randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,first", [(5, 2048, 6144, True), (640, 1536, 8192, True), (897, 2048, 6144, False),
                                         (1312, 1501, 2048, True), (1309, 1501, 2048, False)])
@pytest.mark.parametrize("bits,sym,mx,group", [(8, False, False, 128), (4, False, False, 64), (4, True, True, 32)],
                         ids=["8asym", "4asym", "mx"])
def test_same_bits(bits, sym, mx, group, m, n, k, first, dev):
    from lemoq import _hip
    from lemoq.kernels.dequant_gemm import _weight_first, dequant_gemm_separate
    from lemoq.quant.formats import format_id
    from lemoq.quant.linear import QuantLinear

    print("case: weight first lines %d sym=%s mx=%s m=%d n=%d k=%d" % (bits, sym, mx, m, n, k), flush=True)
    fmt = format_id(bits, sym, mx)
    assert _weight_first(fmt, m, n, k) == first
    lin = QuantLinear(randn(n, k, seed=n + k, std=0.02).to(dev), group_size=group, symmetric=sym,
                      scheme="mxfp4" if mx else "w%da16" % bits)
    x = randn(m, k, seed=m + k).to(torch.float16).to(dev)
    zero = None if sym else lin.zero
    y = torch.full((m, n), float("nan"), dtype=torch.float16, device=dev)
    P = _hip.ptr
    _hip.call("lemoq_gemm_q", P(x), m, k, k, P(lin.packed), fmt, P(lin.scale), P(zero), n, lin.group_size, P(y), n,
              _hip.stream_of(dev))
    got = dequant_gemm_separate(x, lin.packed, lin.scale, zero, group_size=lin.group_size, bits=bits, symmetric=sym,
                                mxfp4=mx)
    torch.cuda.synchronize()
    assert torch.equal(got, y)

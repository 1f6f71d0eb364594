"""Symmetric 8-bit weights that come with a zero tensor (rtn's output always has one).

Groups of 64 and 128 run ``lemoq_gemm_q``'s LEMOQ_QFMT_W8, which equals
``lemoq_gemm_w8`` bit for bit; groups of 32 and 96, which it does not take, are
dequantised first: the fp16 GEMM on the same weights, bit for bit."""

from __future__ import annotations

import pytest
import torch

from helpers import randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(1, 100, 192), (33, 136, 384), (140, 1100, 3456), (520, 6144, 384)])
@pytest.mark.parametrize("group", [32, 64, 96, 128])
def test_symmetric_w8_with_a_zero_tensor(m, n, k, group, dev):
    from lemoq import _hip
    from lemoq.kernels.dequant_gemm import dequant_gemm_separate, linear_f16
    from lemoq.quant.formats import QFMT_W8, dequantize
    from lemoq.quant.rtn import quantize_rtn

    if k % group:
        pytest.skip("no whole number of groups")
    print("case: w8 with zero m=%d n=%d k=%d g=%d" % (m, n, k, group), flush=True)
    q = quantize_rtn(randn(n, k, seed=n + k, std=0.02).to(dev), bits=8, group_size=group)
    x = randn(m, k, seed=m + k).to(torch.float16).to(dev)
    got = dequant_gemm_separate(x, q["packed"], q["scale_f16"], q["zero_f16"], group_size=group)
    w = dequantize(q["packed"], q["scale_f16"], None, fmt=QFMT_W8, group_size=group, k_out=k, dtype=torch.float16)
    want = linear_f16(x, w)
    if group % 64 == 0:
        w8 = dequant_gemm_separate(x, q["packed"], q["scale_f16"], group_size=group)
        assert torch.equal(got, w8)
        y = torch.full((m, n), float("nan"), dtype=torch.float16, device=dev)
        P = _hip.ptr
        _hip.call("lemoq_gemm_q", P(x), m, k, k, P(q["packed"]), QFMT_W8, P(q["scale_f16"]), None, n, group, P(y), n,
                  _hip.stream_of(dev))
        assert torch.equal(got, y)
    torch.cuda.synchronize()
    assert torch.equal(got, want)

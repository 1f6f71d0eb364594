"""``dequant_gemm_separate``'s choice of a launch, on the CPU with the C call stubbed:
every format, scale type and group that the argument rules accept reaches an entry
whose own rules take it (lemoq_hip.h: lemoq_gemm_w8 groups of 64, lemoq_gemm_q
groups of 64 for LEMOQ_QFMT_W8 and of 32 for the others, MXFP4 of 32 alone)."""

from __future__ import annotations

import pytest
import torch

from lemoq import _hip
from lemoq.kernels import dequant_gemm as dg
from lemoq.quant import formats

M, N, K = 3, 40, 1152  # a multiple of 64, 96 and 128


@pytest.fixture
def calls(monkeypatch):
    got = []
    monkeypatch.setattr(_hip, "require_rocm", lambda *a, **k: None)
    monkeypatch.setattr(_hip, "stream_of", lambda *a: 0)
    monkeypatch.setattr(_hip, "call", lambda name, *a: got.append((name, a)))
    return got


def _case(bits: int, symmetric: bool, mxfp4: bool, group: int, scale_dtype, with_zero: bool):
    code = torch.uint8 if bits == 4 or not symmetric else torch.int8
    q = torch.zeros((N, K if bits == 8 else K // 2), dtype=code)
    scale = torch.ones((N, K // group), dtype=torch.uint8 if mxfp4 else scale_dtype)
    return q, scale, torch.zeros((N, K // group), dtype=scale_dtype) if with_zero else None


@pytest.mark.parametrize("bits,symmetric,mxfp4", [(8, True, False), (8, False, False), (4, True, False),
                                                  (4, False, False), (4, True, True)])
@pytest.mark.parametrize("group", [16, 32, 48, 64, 96, 128])
@pytest.mark.parametrize("scale_dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("with_zero", [False, True])
def test_entry_takes_what_it_is_given(bits, symmetric, mxfp4, group, scale_dtype, with_zero, calls):
    if group % (16 if bits == 8 else 32) or (mxfp4 and (group != 32 or with_zero)) or (not symmetric and not with_zero):
        pytest.skip("refused by the argument rules")
    q, scale, zero = _case(bits, symmetric, mxfp4, group, scale_dtype, with_zero)
    plain_w8 = bits == 8 and symmetric and zero is None and scale_dtype == torch.float16
    x = torch.zeros((M, K), dtype=torch.float16)
    kw = dict(group_size=group, bits=bits, symmetric=symmetric, mxfp4=mxfp4)
    if plain_w8 and group % 64:
        with pytest.raises(NotImplementedError, match="group_size"):
            dg.dequant_gemm_separate(x, q, scale, zero, **kw)
        return
    assert dg.dequant_gemm_separate(x, q, scale, zero, **kw).shape == (M, N)
    names = [name for name, _ in calls]
    if plain_w8:
        assert names == ["lemoq_gemm_w8"]
        return
    step = 64 if bits == 8 and symmetric else 32
    in_gemm = (mxfp4 or scale_dtype == torch.float16) and group % step == 0
    assert names == (["lemoq_gemm_q"] if in_gemm else ["lemoq_dequant_q", "lemoq_gemm_f16"])
    if in_gemm:
        fmt, g = calls[0][1][5], calls[0][1][9]
        assert fmt == formats.format_id(bits, symmetric, mxfp4) and g == group


def test_refusals_of_a_half_stage_say_what_they_need(calls):
    """2000 MXFP4 inputs pad to 2016, which is no multiple of 64: several tokens are refused."""
    rows = torch.zeros((M, 2016), dtype=torch.float16)
    q, scale = torch.zeros((N, 1008), dtype=torch.uint8), torch.ones((N, 63), dtype=torch.uint8)
    with pytest.raises(NotImplementedError, match=r"padded_in % 64 == 0, got 2016"):
        dg.dequant_gemm_separate(rows, q, scale, group_size=32, bits=4, mxfp4=True)
    with pytest.raises(NotImplementedError, match=r"K % 64 == 0, got 2016"):
        dg.linear_f16(rows, torch.zeros((N, 2016), dtype=torch.float16))
    assert not calls


@pytest.mark.parametrize("m,n,k,first", [(1024, 1792, 6144, True), (1024, 1793, 6144, False), (1, 2048, 8192, True),
                                         (1, 2048, 4096, False), (896, 2048, 6144, True), (897, 2048, 6144, False),
                                         (1312, 1501, 2048, True), (1309, 1501, 2048, False), (2052, 1501, 2048, True),
                                         (2053, 1501, 2048, False), (1700, 1501, 1024, False), (1700, 1504, 2048, False),
                                         (1, 2056, 8192, False), (2048, 2047, 2048, True), (2049, 2047, 2048, False), (2048, 2048, 2048, False),
                                         (2, 1024, 3072, True), (2, 1024, 2048, False)])
def test_weight_first_lines(m, n, k, first):
    """Both sides of each line of the rule for narrow outputs; never for the formats that
    dequantise in packed fp16."""
    for fmt in (formats.QFMT_W8_ASYM, formats.QFMT_W4_ASYM, formats.QFMT_MXFP4):
        assert dg._weight_first(fmt, m, n, k) == first
    for fmt in (formats.QFMT_W8, formats.QFMT_W4):
        assert not dg._weight_first(fmt, m, n, k)

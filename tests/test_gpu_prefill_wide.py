"""Edges of the direct-load w8 main loop (csrc/gemm_wide.h) in the dense and grouped GEMMs.

K of one, two and three stages (shorter than the ring), scale rows that do and
do not move as 16-byte chunks, more scale groups than fit in LDS at once (they
are reloaded on the way), row tiles of every fragment count with their
remainders, ragged columns, gathered rows in every block shape.  Oracle and
bounds as in test_gpu_prefill_gemm.py: fp64 products of the fp16 weights, one
fp16 ulp plus 3e-5 * sum|x||w| for the fp32 sums.

The gate/up epilogue's SiLU is checked for every finite fp16 gate.
"""

from __future__ import annotations

import pytest
import torch

from helpers import assert_close, randn
from oracle import ops
from oracle import quant as oq

pytestmark = pytest.mark.gpu


def _q8(w: torch.Tensor, group: int):
    q = oq.rtn_quantize_w8(w.numpy(), group)
    return torch.from_numpy(q["codes_padded"]), torch.from_numpy(q["scale_f16"])


def _ulp16(r: torch.Tensor) -> torch.Tensor:
    return torch.exp2(torch.floor(torch.log2(r.double().abs().clamp_min(2.0 ** -14))) - 10)


CASES = [
    (1, 100, 64, 64, False),        # one stage, one row, ragged columns
    (140, 1024, 64, 64, False),     # one stage, rows that leave through the LDS its loads went to, 32-row tiles
    (700, 2048, 64, 64, True),      # ... 64-row tiles
    (4096, 6144, 64, 64, False),    # ... 128-row tiles of 256 columns
    (33, 136, 128, 64, True),       # two stages; two fragments, one of one row
    (97, 200, 192, 64, False),      # three stages, three scale groups (no 16-byte chunks)
    (65, 320, 512, 64, True),       # eight groups
    (300, 130, 4352, 64, False),    # 68 groups: reloaded twice
    (700, 6144, 256, 128, True),    # 96-row tiles of 256 columns
    (1100, 6016, 2112, 64, False),  # 128-row tiles of 256 columns, 33 groups, ragged rows and columns
    (520, 6144, 256, 64, True),     # 128 x 128 tiles
    (129, 1001, 128, 64, True),     # unaligned rows out, 32-row tiles
    (600, 4099, 64, 64, False),     # ... 64-row tiles
    (1030, 4099, 64, 64, False),    # ... 96-row tiles of 256 columns
    (1500, 4099, 64, 64, True),     # ... 128 x 128 tiles
]


@pytest.mark.parametrize("m,n,k,group,gather", CASES, ids=["%dx%dx%d-g%d%s" % (c[:4] + ("-gather" if c[4] else "",))
                                                           for c in CASES])
def test_gemm_w8_edges(m, n, k, group, gather, dev):
    from lemoq import _hip

    print("case: gemm_w8 edge m=%d n=%d k=%d g=%d gather=%s" % (m, n, k, group, gather), flush=True)
    codes, scale = _q8(randn(n, k, seed=n + k, std=0.02), group)
    rows = m + 9 if gather else m
    x = randn(rows, k, seed=m + k).to(torch.float16)
    idx = torch.randperm(rows, generator=torch.Generator().manual_seed(m))[:m].to(torch.int32)
    xd, cd, sd, idd = x.to(dev), codes.to(dev), scale.to(dev), idx.to(dev)
    y = torch.full((m, n), float("nan"), dtype=torch.float16, device=dev)
    _hip.call("lemoq_gemm_w8", _hip.ptr(xd), m, k, k, _hip.ptr(idd) if gather else None, _hip.ptr(cd), _hip.ptr(sd),
              n, group, _hip.ptr(y), n, None, 0, _hip.stream_of(dev))
    torch.cuda.synchronize()
    xg = x[idx.long()] if gather else x
    ref = ops.linear_separate_w8(xg, codes, scale, group)
    absdot = xg.double().abs() @ ops.dequant_weight_f16(codes, scale, group).double().abs().t()
    err = (y.cpu().double() - ref.double()).abs()
    assert bool((err <= _ulp16(ref) + 3e-5 * absdot).all()), float(err.max())


MOE = [
    (1, 4224, 64, 8, 64),    # one token (thin blocks), 66 groups
    (40, 4224, 64, 32, 64),  # half-width blocks, 66 groups
    (70, 64, 96, 32, 64),    # one stage; gate/up columns end inside a block
    (130, 192, 64, 3, 64),   # three groups; every expert with two uneven tiles
]


@pytest.mark.parametrize("T,H,F,E,group", MOE, ids=["T%d-H%d-F%d-E%d-g%d" % c for c in MOE])
def test_moe_prefill_edges(T, H, F, E, group, dev):
    from lemoq import _hip

    print("case: moe_prefill edge T=%d H=%d F=%d E=%d g=%d" % (T, H, F, E, group), flush=True)
    K = min(2, E)
    F64 = -(-F // 64) * 64  # down's reduction width: whole stages
    g = torch.Generator().manual_seed(T + H)
    x = torch.randn((T, H), generator=g).to(torch.float16)
    gu_c = torch.randint(-127, 128, (E, 2 * F, H), generator=g, dtype=torch.int8)
    dn_c = torch.randint(-127, 128, (E, H, F64), generator=g, dtype=torch.int8)
    gu_s = ((torch.rand((E, 2 * F, H // group), generator=g) + 0.5) * (0.035 / 127)).to(torch.float16)
    dn_s = ((torch.rand((E, H, F64 // group), generator=g) + 0.5) * (0.035 / 127)).to(torch.float16)
    ti = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(T)])
    tw = torch.rand((T, K), generator=g)
    P, st, lib = _hip.ptr, _hip.stream_of(dev), _hip.load()
    pairs = T * K
    mt = int(lib.lemoq_moe_prefill_max_tiles(pairs, E))
    i32 = dict(dtype=torch.int32, device=dev)
    d = [t.to(dev) for t in (x, gu_c, gu_s, dn_c, dn_s, ti, tw)]
    tok, src, off = torch.empty((pairs,), **i32), torch.empty((pairs,), **i32), torch.empty((E + 1,), **i32)
    tiles = torch.empty((mt, 4), **i32)
    pw = torch.empty((pairs,), dtype=torch.float16, device=dev)
    act = torch.zeros((pairs, F64), dtype=torch.float16, device=dev)
    gu_out = torch.full((pairs, F), float("nan"), dtype=torch.float16, device=dev)
    y = torch.full((pairs, H), float("nan"), dtype=torch.float16, device=dev)
    _hip.call("lemoq_moe_prefill_sort", P(d[5]), P(d[6]), T, K, E, P(tok), P(src), P(pw), P(off), P(tiles), mt, st)
    _hip.call("lemoq_moe_prefill_gate_up", P(d[0]), H, P(tok), P(tiles), mt, P(d[1]), P(d[2]), F, group, P(gu_out),
              st)
    act[:, :F] = gu_out
    _hip.call("lemoq_moe_prefill_down", P(act), F64, P(src), P(pw), P(tiles), mt, P(d[3]), P(d[4]), H, group, P(y),
              st)
    torch.cuda.synchronize()
    live = tiles.cpu()
    live = live[live[:, 0] >= 0]
    assert bool((live[:, 3] == live.shape[0]).all())  # every used row holds their number
    act_ref = torch.empty((pairs, F), dtype=torch.float16)
    srcs = src.cpu().long()
    experts = ti.reshape(-1)[srcs]
    for e in range(E):
        rows = (experts == e).nonzero().reshape(-1)
        gu = ops.linear_separate_w8(x[srcs[rows] // K], gu_c[e], gu_s[e], group)
        act_ref[rows] = torch.nn.functional.silu(gu[:, :F]) * gu[:, F:]
    assert_close(gu_out.cpu(), act_ref, what="gate_up")
    a = act.cpu()
    for e in range(E):
        rows = (experts == e).nonzero().reshape(-1)
        ref = ops.linear_separate_w8(a[rows], dn_c[e], dn_s[e], group) * tw.reshape(-1)[srcs[rows], None].half()
        assert_close(y.cpu()[srcs[rows]], ref, what="down expert %d" % e)


def test_gate_up_silu_every_gate(dev):
    """act = silu(gate) for every finite fp16 gate (up = 1): equal to the fp32
    quotient rounded to fp16, but for at most one gate whose exact value lies
    beside the middle of two fp16 values."""
    from lemoq import _hip

    gates = torch.arange(0x7C00, dtype=torch.int32)
    gates = torch.cat((gates, gates | 0x8000)).to(torch.uint16).view(torch.float16)
    T, H, F = int(gates.numel()), 64, 32
    P, st = _hip.ptr, _hip.stream_of(dev)
    x = torch.zeros((T, H), dtype=torch.float16)
    x[:, 0], x[:, 1] = gates, 1.0
    codes = torch.zeros((1, 2 * F, H), dtype=torch.int8)
    codes[0, :F, 0] = 1  # gate rows pick x[0], up rows x[1]
    codes[0, F:, 1] = 1
    i32 = dict(dtype=torch.int32, device=dev)
    begins = torch.arange(0, T, 128)
    tiles = torch.stack((torch.zeros_like(begins), begins, (begins + 128).clamp(max=T), torch.zeros_like(begins)), 1)
    td = tiles.to(**i32).contiguous()
    tok = torch.arange(T, **i32)
    scale = torch.ones((1, 2 * F, 1), dtype=torch.float16, device=dev)
    act = torch.empty((T, F), dtype=torch.float16, device=dev)
    xd, cd = x.to(dev), codes.to(dev)
    _hip.call("lemoq_moe_prefill_gate_up", P(xd), H, P(tok), P(td), int(begins.numel()), P(cd), P(scale), F, 64,
              P(act), st)
    torch.cuda.synchronize()
    got = act.cpu()
    assert torch.equal(got, got[:, :1].expand_as(got))
    g = gates.float()
    want = (g / (1.0 + torch.exp(-g))).to(torch.float16)
    off = (got[:, 0].view(torch.int16) != want.view(torch.int16)) & ~((got[:, 0] == 0) & (want == 0))
    exact = gates.double() / (1.0 + torch.exp(-gates.double()))
    ulp = _ulp16(want)
    assert int(off.sum()) <= 1, gates[off].tolist()
    assert bool(((got[:, 0].double() - exact).abs() <= ulp * (0.5 + 1e-3)).all())


def test_gate_up_silu_bits(dev):
    """act = fp16(g / (1 + exp(-g))) in fp32, bit for bit, for all 65536 fp16 gates:
    finite ones, and infinite and NaN gates (which only the gate rows' scales make, so
    that the up rows stay 1)."""
    from lemoq import _hip

    finite = torch.arange(0x7C00, dtype=torch.int32)
    x0 = torch.cat((finite, finite | 0x8000)).to(torch.uint16).view(torch.float16)
    T, H, F = int(x0.numel()), 64, 32
    P, st = _hip.ptr, _hip.stream_of(dev)
    x = torch.zeros((T, H), dtype=torch.float16)
    x[:, 0], x[:, 1] = x0, 1.0
    codes = torch.zeros((1, 2 * F, H), dtype=torch.int8)
    codes[0, :F, 0] = 1  # gate rows pick x[0], up rows x[1]
    codes[0, F:, 1] = 1
    scale = torch.ones((1, 2 * F, 1), dtype=torch.float16)
    codes[0, F - 2, 0], scale[0, F - 2, 0] = 127, 512.0  # gates beyond 1 overflow to +-inf
    scale[0, F - 1, 0] = float("nan")
    i32 = dict(dtype=torch.int32, device=dev)
    begins = torch.arange(0, T, 128)
    tiles = torch.stack((torch.zeros_like(begins), begins, (begins + 128).clamp(max=T), torch.zeros_like(begins)), 1)
    td = tiles.to(**i32).contiguous()
    tok = torch.arange(T, **i32)
    act = torch.empty((T, F), dtype=torch.float16, device=dev)
    xd, cd, sd = x.to(dev), codes.to(dev), scale.to(dev)
    _hip.call("lemoq_moe_prefill_gate_up", P(xd), H, P(tok), P(td), int(begins.numel()), P(cd), P(sd), F, 64,
              P(act), st)
    gates = torch.stack((xd[:, 0], (xd[:, 0].double() * (127 * 512.0)).to(torch.float16), xd[:, 0] * float("nan")), 1)
    g = gates.float() + 0.0  # a sum from 0 has no -0
    want = (g / (1.0 + torch.exp(-g))).to(torch.float16)
    got = act[:, F - 3:]
    assert bool(gates.isinf().any()) and bool(gates.isnan().any())
    same = (got.view(torch.int16) == want.view(torch.int16)) | (got.isnan() & want.isnan())
    assert bool(same.all()), gates[~same].tolist()[:8]


Q_CASES = [  # bits, symmetric, mxfp4, group
    (8, False, False, 32), (8, False, False, 128), (4, True, False, 32), (4, True, False, 96), (4, True, False, 128),
    (4, False, False, 64), (4, False, False, 128), (4, True, True, 32),
]
Q_SHAPES = [(1, 100, 192), (33, 136, 384), (140, 1100, 3456), (520, 6144, 192), (1100, 6016, 384)]


@pytest.mark.parametrize("m,n,k", Q_SHAPES, ids=["%dx%dx%d" % s for s in Q_SHAPES])
@pytest.mark.parametrize("bits,sym,mx,group", Q_CASES, ids=["%d%s%s-g%d" % (c[0], "" if c[1] else "asym",
                                                                            "mx" if c[2] else "", c[3])
                                                            for c in Q_CASES])
def test_gemm_q_equals_dequantised_weight(bits, sym, mx, group, m, n, k, dev):
    """The GEMM on the codes against the fp16 GEMM on the same format's
    dequantised weight (lemoq_dequant_q): the same fp16 weights, so the fp64
    products of those weights bound it as in test_gemm_w8_edges."""
    from lemoq import _hip
    from lemoq.quant.formats import dequantize, format_id
    from lemoq.quant.linear import QuantLinear

    if k % group:
        k += group - k % group
        k += (64 - k % 64) % 64 if (k + (64 - k % 64) % 64) % group == 0 else 0
    if k % 64 or k % group:
        pytest.skip("no whole number of groups and stages")
    print("case: gemm_q %d sym=%s mx=%s g=%d m=%d n=%d k=%d" % (bits, sym, mx, group, m, n, k), flush=True)
    lin = QuantLinear(randn(n, k, seed=n + k, std=0.02).to(dev), group_size=group, symmetric=sym,
                      scheme="mxfp4" if mx else "w%da16" % bits)
    fmt = format_id(bits, sym, mx)
    x = randn(m, k, seed=m + k).to(torch.float16).to(dev)
    y = torch.full((m, n), float("nan"), dtype=torch.float16, device=dev)
    _hip.call("lemoq_gemm_q", _hip.ptr(x), m, k, k, _hip.ptr(lin.packed), fmt, _hip.ptr(lin.scale),
              None if sym else _hip.ptr(lin.zero), n, lin.group_size, _hip.ptr(y), n, _hip.stream_of(dev))
    w = dequantize(lin.packed, lin.scale, lin.zero, fmt=fmt, group_size=lin.group_size, k_out=k,
                   dtype=torch.float16)
    torch.cuda.synchronize()
    ref64 = x.double() @ w.double().t()
    absdot = x.double().abs() @ w.double().abs().t()
    err = (y.double() - ref64).abs()
    assert bool((err <= _ulp16(ref64.to(torch.float16)).to(dev) + 3e-5 * absdot).all()), float(err.max())


@pytest.mark.parametrize("m,n,k", [(3, 64, 4096), (1830, 1001, 3072), (1793, 1001, 2048), (3073, 1500, 2048),
                                   (1793, 1024, 3072), (3072, 1500, 2048), (40, 1032, 4096)])
@pytest.mark.parametrize("bits,sym,mx,group", [(8, False, False, 128), (4, False, False, 64), (4, True, True, 32),
                                               (4, True, False, 128)],
                         ids=["8asym", "4asym", "mx", "4sym"])
def test_weight_first_same_bits(bits, sym, mx, group, m, n, k, dev):
    """Both sides of the rule for narrow outputs give the codes' GEMM bit for bit
    (the same fp16 weights, fp32 sums over k in the same order)."""
    from lemoq import _hip
    from lemoq.kernels.dequant_gemm import _weight_first, dequant_gemm_separate
    from lemoq.quant.formats import format_id
    from lemoq.quant.linear import QuantLinear

    fmt = format_id(bits, sym, mx)
    first = (n <= 1001 or m == 3073) and not (bits == 4 and sym and not mx)
    assert _weight_first(fmt, m, n, k) == first
    print("case: weight first %d sym=%s mx=%s m=%d n=%d k=%d" % (bits, sym, mx, m, n, k), flush=True)
    lin = QuantLinear(randn(n, k, seed=n + k, std=0.02).to(dev), group_size=group, symmetric=sym,
                      scheme="mxfp4" if mx else "w%da16" % bits)
    x = randn(m, k, seed=m + k).to(torch.float16).to(dev)
    zero = None if sym else lin.zero
    y = torch.full((m, n), float("nan"), dtype=torch.float16, device=dev)
    _hip.call("lemoq_gemm_q", _hip.ptr(x), m, k, k, _hip.ptr(lin.packed), fmt, _hip.ptr(lin.scale), _hip.ptr(zero), n,
              lin.group_size, _hip.ptr(y), n, _hip.stream_of(dev))
    got = dequant_gemm_separate(x, lin.packed, lin.scale, zero, group_size=lin.group_size, bits=bits, symmetric=sym,
                                mxfp4=mx)
    torch.cuda.synchronize()
    assert torch.equal(got, y)

"""One row through the last layer of a prefill: the bits of the multi-token launches.

- ``lemoq_gemm_w8`` of one row against the first row of the same product over two
  (the tiles' main loop), with and without a gather and a residual.
- ``lemoq_moe_gate_up_w8_dq`` (and its routed form) + ``lemoq_moe_down_w8_dq``
  against the sort, the grouped GEMMs and the combine of the same row.
- ``prefill_prompt``: its logits with the MoE block in the one-row form and in
  the grouped launches.

All bit for bit.  K and F around the row kernels' stages of 512, rings of them and
the chunks of 32 in them; columns around a wave's 32 and on both sides of the
rule that leaves wide outputs to the tiles.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _w8(g: torch.Generator, *shape: int, group: int, dev) -> tuple[torch.Tensor, torch.Tensor]:
    codes = torch.randint(-127, 128, shape, generator=g, dtype=torch.int8)
    scale = ((torch.rand((*shape[:-1], shape[-1] // group), generator=g) + 0.5) * (0.035 / 127)).to(torch.float16)
    return codes.to(dev), scale.to(dev)


@pytest.mark.parametrize("K,N,group", [(64, 1, 64), (512, 33, 128), (576, 64, 64), (1024, 100, 1024), (1088, 31, 64),
                                       (1600, 1001, 320), (2048, 2048, 128), (4352, 96, 64), (64, 16384, 64), (64, 16385, 64)])
@pytest.mark.parametrize("extra", [False, True], ids=["plain", "gather-residual"])
def test_gemm_w8_one_row(K, N, group, extra, dev):
    from lemoq import _hip

    print("case: gemm_w8 one row K=%d N=%d g=%d %s" % (K, N, group, extra), flush=True)
    g = torch.Generator().manual_seed(K + N)
    codes, scale = _w8(g, N, K, group=group, dev=dev)
    x = torch.randn((5, K), generator=g).to(torch.float16).to(dev)
    rows = torch.tensor([3, 1], dtype=torch.int32, device=dev)
    res = torch.randn((2, N), generator=g).to(torch.float16).to(dev)
    P, st = _hip.ptr, _hip.stream_of(dev)
    got = []
    for m in (1, 2):
        y = torch.full((2, N), float("nan"), dtype=torch.float16, device=dev)
        _hip.call("lemoq_gemm_w8", P(x), m, K, K, P(rows) if extra else None, P(codes), P(scale), N, group, P(y), N,
                  P(res) if extra else None, N, st)
        got.append(y)
    torch.cuda.synchronize()
    assert bool(got[1].isfinite().all()) and bool(got[0][1].isnan().all())
    assert torch.equal(got[0][0], got[1][0])


def _padded(t: torch.Tensor, cols: int) -> torch.Tensor:
    return torch.nn.functional.pad(t, (0, cols - t.shape[-1])).contiguous()


@pytest.mark.parametrize("H,F,E,K,group", [(2048, 1024, 64, 8, 128), (512, 192, 100, 8, 64), (1088, 320, 7, 3, 64),
                                           (4096, 64, 255, 1, 64), (256, 8192, 5, 5, 128), (1024, 288, 16, 2, 32),
                                           (1040, 80, 5, 5, 16)])
@pytest.mark.parametrize("norm", [False, True])
def test_moe_row_equals_grouped(H, F, E, K, group, norm, dev):
    """Groups of 16 and 32, and widths that are no whole stage, which the grouped
    GEMMs do not take, run there as groups of 64 (the scales in fours and twos)
    and zero columns."""
    from lemoq import _hip

    print("case: moe row H=%d F=%d E=%d k=%d g=%d norm=%s" % (H, F, E, K, group, norm), flush=True)
    g = torch.Generator().manual_seed(H + F + E)
    wide = max(group, 64)
    Hp, Fp = -(-H // 64) * 64, -(-F // 64) * 64

    def weight(rows: int, cols: int, padded: int):
        codes, scale = _w8(g, E, rows, padded, group=wide, dev=dev)
        codes[..., cols:] = 0
        return (codes, scale), (codes[..., :cols].contiguous(),
                                scale.repeat_interleave(wide // group, -1)[..., : cols // group].contiguous())

    (gu_p, gus_p), (gu, gus) = weight(2 * F, H, Hp)
    (dn_p, dns_p), (dn, dns) = weight(H, F, Fp)
    x, res = (torch.randn((H,), generator=g).to(torch.float16).to(dev) for _ in range(2))
    logits = torch.randn((E,), generator=g).to(torch.float16).to(dev)
    P, st, lib = _hip.ptr, _hip.stream_of(dev), _hip.load()
    f16, i32 = dict(dtype=torch.float16, device=dev), dict(dtype=torch.int32, device=dev)
    top_w, top_i = torch.empty((K,), device=dev), torch.empty((K,), dtype=torch.int64, device=dev)
    _hip.call("lemoq_route_topk", P(logits), 1, 1, E, E, K, int(norm), P(top_w), P(top_i), st)

    def row(routed: bool) -> tuple:
        act, w, ids = torch.full((K, F), float("nan"), **f16), torch.empty((K,), **f16), top_i.clone()
        if routed:
            ids.fill_(-1)
            _hip.call("lemoq_moe_gate_up_w8_routed_dq", P(x), P(gu), P(gus), P(logits), K, int(norm), E, F, H, group,
                      P(act), P(ids), P(w), st)
        else:
            _hip.call("lemoq_moe_gate_up_w8_dq", P(x), P(gu), P(gus), P(top_i), P(top_w), K, E, F, H, group, P(act), P(w),
                      st)
        out = res.clone()  # the residual may alias the output
        _hip.call("lemoq_moe_down_w8_dq", P(act), P(dn), P(dns), P(ids), P(w), K, E, H, F, group, P(out), P(out), st)
        torch.cuda.synchronize()
        return act, w, ids, out

    act, w, ids, out = row(False)
    for a, b in zip(row(True), (act, w, top_i, out)):
        assert torch.equal(a, b)
    mt = int(lib.lemoq_moe_prefill_max_tiles(K, E))
    tok, src, off = torch.empty((K,), **i32), torch.empty((K,), **i32), torch.empty((E + 1,), **i32)
    tiles, pw = torch.empty((mt, 4), **i32), torch.empty((K,), **f16)
    xp = _padded(x, Hp)
    gact = torch.full((K, F), float("nan"), **f16)
    _hip.call("lemoq_moe_prefill_sort", P(top_i), P(top_w), 1, K, E, P(tok), P(src), P(pw), P(off), P(tiles), mt, st)
    if F % 32 == 0:
        _hip.call("lemoq_moe_prefill_gate_up", P(xp), Hp, P(tok), P(tiles), K, P(gu_p), P(gus_p), F, wide, P(gact), st)
        torch.cuda.synchronize()
        assert torch.equal(act[src.long()], gact)
    order = src.long()
    assert torch.equal(w[order], pw)
    if H % 32 == 0:
        ap = _padded(act[order], Fp)
        y, want = torch.full((K, H), float("nan"), **f16), res.clone()
        _hip.call("lemoq_moe_prefill_down", P(ap), Fp, P(src), P(pw), P(tiles), K, P(dn_p), P(dns_p), H, wide, P(y), st)
        _hip.call("lemoq_moe_prefill_combine", P(y), P(top_i), 1, K, H, P(want), P(want), st)
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("T", [2, 75])
def test_prefill_last_row_bits(T, dev, monkeypatch):
    """The MoE block's one-row launches of a prefill against the grouped ones, which
    stand in for them call by call."""
    from lemoq import _hip
    from lemoq.kernels.rope import rotary_cos_sin
    from lemoq.model.olmoe import OlmoeShape, OlmoeW8Weights
    from lemoq.model.prefill import prefill_prompt

    print("case: prefill last row bits T=%d" % T, flush=True)
    shape = OlmoeShape(hidden=2048, heads=16, head_dim=128, layers=2, num_experts=16, top_k=4, ffn=256, vocab=4096)
    wts = OlmoeW8Weights.random(shape, seed=T, device=dev)
    S = T + 3
    cos, sin = (t.to(dev).contiguous() for t in rotary_cos_sin(torch.arange(S), shape.head_dim, shape.rope_theta))
    tokens = torch.randint(0, shape.vocab, (T,), generator=torch.Generator().manual_seed(T)).to(dev)
    call, lib, P = _hip.call, _hip.load(), _hip.ptr
    i32, f16 = dict(dtype=torch.int32, device=dev), dict(dtype=torch.float16, device=dev)
    K, E = shape.top_k, shape.num_experts
    mt = int(lib.lemoq_moe_prefill_max_tiles(K, E))
    tok, src, off = torch.empty((K,), **i32), torch.empty((K,), **i32), torch.empty((E + 1,), **i32)
    tiles, pw, y = torch.empty((mt, 4), **i32), torch.empty((K,), **f16), torch.empty((K, shape.hidden), **f16)
    seen = []

    def grouped(name, *a):
        if name == "lemoq_moe_gate_up_w8_dq":
            x, codes, scale, ids, w32, k, e, F, H, g, act, _, s = a
            call("lemoq_moe_prefill_sort", ids, w32, 1, k, e, P(tok), P(src), P(pw), P(off), P(tiles), mt, s)
            call("lemoq_moe_prefill_gate_up", x, H, P(tok), P(tiles), k, codes, scale, F, g, act, s)
            seen.append((ids, k))
        elif name == "lemoq_moe_down_w8_dq":
            act, codes, scale, ids, _, k, _, H, F, g, res, out, s = a
            call("lemoq_moe_prefill_down", act, F, P(src), P(pw), P(tiles), k, codes, scale, H, g, P(y), s)
            call("lemoq_moe_prefill_combine", P(y), ids, 1, k, H, res, out, s)
        else:
            call(name, *a)

    got = []
    for fn in (call, grouped):
        kv = [{n: torch.zeros((shape.heads, S, 128), **f16) for n in ("k", "v")} for _ in range(shape.layers)]
        logits = torch.empty((shape.vocab,), **f16)
        monkeypatch.setattr(_hip, "call", fn)
        prefill_prompt(wts, tokens, kv, cos, sin, S, logits)
        torch.cuda.synchronize()
        got.append(logits)
    assert len(seen) == 1
    assert torch.equal(got[0], got[1])

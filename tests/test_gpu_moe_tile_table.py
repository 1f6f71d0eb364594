"""Tile tables of a caller's own in the grouped MoE GEMMs: the fourth column is a hint
and loses no tile, whatever it holds, unused rows (expert -1) between used ones among
them; in every block shape.  Against the same table with zeros there, bit for bit, and
every row of every used tile written."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ntiles,F", [(5, 96), (40, 128), (70, 1024)], ids=["thin", "half", "wide"])
def test_fourth_column_is_a_hint(ntiles, F, dev):
    from lemoq import _hip

    print("case: tile table %d tiles F=%d" % (ntiles, F), flush=True)
    H, E, rows = 128, 3, 32
    g = torch.Generator().manual_seed(ntiles)
    used = [i for i in range(ntiles) if i % 7 != 3]  # every seventh row unused
    pairs = rows * len(used)
    x = torch.randn((pairs, H), generator=g).to(torch.float16).to(dev)
    gu = torch.randint(-127, 128, (E, 2 * F, H), generator=g, dtype=torch.int8).to(dev)
    dn = torch.randint(-127, 128, (E, H, 128), generator=g, dtype=torch.int8).to(dev)
    gus, dns = (torch.full((E, n, k // 64), 1e-3, dtype=torch.float16, device=dev) for n, k in ((2 * F, H), (H, 128)))
    tok = torch.arange(pairs, dtype=torch.int32, device=dev)
    w = torch.ones((pairs,), dtype=torch.float16, device=dev)
    xd = torch.randn((pairs, 128), generator=g).to(torch.float16).to(dev)
    P, st = _hip.ptr, _hip.stream_of(dev)
    got = []
    for hint in (0, 1, 3, len(used), ntiles, ntiles + 1, -5, 2 ** 30):
        t = torch.full((ntiles, 4), -1, dtype=torch.int32)
        t[:, 3] = hint
        for n, i in enumerate(used):
            t[i, 0], t[i, 1], t[i, 2] = i % E, rows * n, rows * (n + 1)
        td = t.to(dev)
        act = torch.full((pairs, F), float("nan"), dtype=torch.float16, device=dev)
        y = torch.full((pairs, H), float("nan"), dtype=torch.float16, device=dev)
        _hip.call("lemoq_moe_prefill_gate_up", P(x), H, P(tok), P(td), ntiles, P(gu), P(gus), F, 64, P(act), st)
        _hip.call("lemoq_moe_prefill_down", P(xd), 128, P(tok), P(w), P(td), ntiles, P(dn), P(dns), H, 64, P(y), st)
        torch.cuda.synchronize()
        assert bool(act.isfinite().all()) and bool(y.isfinite().all()), hint
        got.append((act, y))
    for act, y in got[1:]:
        assert torch.equal(act, got[0][0]) and torch.equal(y, got[0][1])

"""A post-attention norm weight that is not 16-byte aligned (a view into a larger
tensor) prefills as an aligned copy of it does, bit for bit."""

from __future__ import annotations

import dataclasses

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 5, 40])
def test_prefill_unaligned_post_norm(T, dev):
    from lemoq.kernels.rope import rotary_cos_sin
    from lemoq.model.olmoe import OlmoeShape, OlmoeW8Weights
    from lemoq.model.prefill import prefill_prompt

    print("case: unaligned post norm T=%d" % T, flush=True)
    shape = OlmoeShape(hidden=512, heads=4, head_dim=128, layers=2, num_experts=16, top_k=4, ffn=256, vocab=4096)
    w = OlmoeW8Weights.random(shape, seed=T, device=dev)
    S = T + 1
    cos, sin = (t.to(dev).contiguous() for t in rotary_cos_sin(torch.arange(S), shape.head_dim, shape.rope_theta))
    tokens = torch.randint(0, shape.vocab, (T,), generator=torch.Generator().manual_seed(T)).to(dev)

    def shifted(t: torch.Tensor) -> torch.Tensor:
        flat = torch.empty((t.numel() + 8,), dtype=t.dtype, device=dev)
        view = flat[1:1 + t.numel()]
        view.copy_(t)
        assert view.data_ptr() % 16 != 0
        return view

    got = []
    for layers in (w.layers, [dataclasses.replace(L, ln_post=shifted(L.ln_post)) for L in w.layers]):
        kv = [{n: torch.zeros((shape.heads, S, 128), dtype=torch.float16, device=dev) for n in ("k", "v")}
              for _ in range(shape.layers)]
        logits = torch.empty((shape.vocab,), dtype=torch.float16, device=dev)
        prefill_prompt(dataclasses.replace(w, layers=layers), tokens, kv, cos, sin, S, logits)
        torch.cuda.synchronize()
        got.append((logits, kv))
    assert torch.equal(got[0][0], got[1][0])
    for a, b in zip(got[0][1], got[1][1]):
        assert torch.equal(a["k"], b["k"]) and torch.equal(a["v"], b["v"])

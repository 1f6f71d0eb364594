"""Weight rows too long for the 32-bit offsets of the direct-load GEMMs: accepted, and
right on both sides of the line.  Bounds as in test_gpu_prefill_wide.py against fp64
products (summed over pieces of K, on the device): one fp16 ulp and 3e-5 * sum|x||w|."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _ulp16(r: torch.Tensor) -> torch.Tensor:
    return torch.exp2(torch.floor(torch.log2(r.abs().clamp_min(2.0 ** -14))) - 10)


def _codes(*shape: int, dev) -> torch.Tensor:
    return torch.randint(-127, 128, shape, dtype=torch.int8, device=dev,
                         generator=torch.Generator(device=dev).manual_seed(shape[-1]))


def _check(got: torch.Tensor, x: torch.Tensor, codes: torch.Tensor, scale: float, what: str) -> None:
    """got (m, n) against x (m, k) @ (fp16(codes * scale))^T, codes (n, k)."""
    y = torch.zeros((x.shape[0], codes.shape[0]), dtype=torch.float64, device=x.device)
    dot = torch.zeros_like(y)
    for k in range(0, x.shape[1], 1 << 18):
        xk = x[:, k:k + (1 << 18)].double()
        w = (codes[:, k:k + (1 << 18)].float() * scale).to(torch.float16).double()
        y += xk @ w.t()
        dot += xk.abs() @ w.abs().t()
    err = (got.double() - y).abs()
    assert bool((err <= _ulp16(y) + 3e-5 * dot).all()), "%s: %g" % (what, float(err.max()))


@pytest.mark.parametrize("K,N,M", [(1 << 23, 130, 3), ((1 << 23) + 64, 130, 3), ((1 << 25) + 64, 130, 2),
                                   ((1 << 23) + 64, 40, 1)])
def test_gemm_w8_long_rows(K, N, M, dev):
    from lemoq import _hip

    print("case: gemm_w8 K=%d N=%d M=%d" % (K, N, M), flush=True)
    s = 2.0 ** -13
    x = torch.randn((M, K), device=dev, generator=torch.Generator(device=dev).manual_seed(M)).to(torch.float16)
    codes = _codes(N, K, dev=dev)
    scale = torch.full((N, 1), s, dtype=torch.float16, device=dev)
    y = torch.full((M, N), float("nan"), dtype=torch.float16, device=dev)
    P = _hip.ptr
    _hip.call("lemoq_gemm_w8", P(x), M, K, K, None, P(codes), P(scale), N, K, P(y), N, None, 0, _hip.stream_of(dev))
    torch.cuda.synchronize()
    _check(y, x, codes, s, "gemm_w8 K=%d" % K)


@pytest.mark.parametrize("K,N", [((1 << 22) + 64, 32), (262208, 16416)], ids=["long-row", "large-expert"])
def test_grouped_long_rows(K, N, dev):
    """gate_up and down of one expert; the gate and up rows have the same codes, so that the
    SiLU's input and its factor are one value."""
    from lemoq import _hip

    print("case: grouped K=%d N=%d" % (K, N), flush=True)
    T, s = 3, 2.0 ** -14
    g = torch.Generator(device=dev).manual_seed(N)
    x = torch.randn((T, K), device=dev, generator=g).to(torch.float16)
    codes = _codes(1, 2 * N, K, dev=dev)
    codes[:, N:] = codes[:, :N]
    P, st = _hip.ptr, _hip.stream_of(dev)
    tiles = torch.tensor([[0, 0, T, 1]], dtype=torch.int32, device=dev)
    tok = torch.arange(T, dtype=torch.int32, device=dev)
    ones = torch.ones((T,), dtype=torch.float16, device=dev)
    y = torch.full((T, N), float("nan"), dtype=torch.float16, device=dev)
    scale = torch.full((1, 2 * N, K // 64), s, dtype=torch.float16, device=dev)
    _hip.call("lemoq_moe_prefill_down", P(x), K, P(tok), P(ones), P(tiles), 1, P(codes), P(scale), N, 64, P(y), st)
    act = torch.full((T, N), float("nan"), dtype=torch.float16, device=dev)
    _hip.call("lemoq_moe_prefill_gate_up", P(x), K, P(tok), P(tiles), 1, P(codes), P(scale), N, 64, P(act), st)
    torch.cuda.synchronize()
    _check(y, x, codes[0, :N], s, "down K=%d" % K)
    v = y.float()
    want = (v / (1.0 + torch.exp(-v))).to(torch.float16) * y  # the same products in the same order
    assert torch.equal(act, want)

"""``QuantLinear`` asks ``fused_available`` on every call, also once the library is
loaded: a subclass that overrides it, and a module function put in its place, decide."""

from __future__ import annotations

import pytest
import torch

from lemoq import _hip
from lemoq.kernels import dequant_gemm
from lemoq.quant.linear import QuantLinear


class _OnDevice:
    """What the dispatch rules look at in a one-token fp16 device tensor."""

    is_cuda, dtype, shape = True, torch.float16, (1, 128)

    def numel(self) -> int:
        return 128


def _linear(cls=QuantLinear):
    return cls.from_packed(torch.zeros((4, 128), dtype=torch.int8), torch.ones((4, 1), dtype=torch.float16),
                           in_features=128, group_size=128)


@pytest.fixture
def loaded(monkeypatch):
    monkeypatch.setattr(_hip, "loaded", lambda: True)
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)


def test_loaded_library_and_device(loaded):
    assert dequant_gemm.fused_available() is True
    assert _linear()._fused_fallback_reason(_OnDevice()) is None


def test_subclass_override_decides(loaded):
    class Without(QuantLinear):
        @property
        def fused_available(self) -> bool:
            return False

    reason = _linear(Without)._fused_fallback_reason(_OnDevice())
    assert reason is not None and reason.startswith("kernel_unavailable(")


def test_module_functions_are_looked_up_at_the_call(loaded, monkeypatch):
    monkeypatch.setattr(dequant_gemm, "fused_available", lambda: False)
    monkeypatch.setattr(dequant_gemm, "unavailable_reason", lambda: "switched off")
    assert _linear()._fused_fallback_reason(_OnDevice()) == "kernel_unavailable(switched off)"
    monkeypatch.setattr(dequant_gemm, "dequant_gemm_separate", lambda x, *a, **k: torch.full((x.shape[0], 4), 7.0))
    assert torch.equal(_linear()(torch.zeros((3, 128), dtype=torch.float16)), torch.full((3, 4), 7.0).half())

"""The workspace of an operator is sized for the device that runs it (the split of K follows its CU count), on the CPU
with the library and the device guard replaced."""
import contextlib

import pytest
import torch

from mindpipe_amd import ops


class _Library:
    def __init__(self):
        self.device, self.asked, self.launched = "current", [], []

    def __getattr__(self, name):
        def call(*args):
            (self.asked if name.endswith("_bytes") else self.launched).append((name, self.device))
            return 256 if name.endswith("_bytes") else 0
        return call


@pytest.mark.parametrize("call", [
    lambda x, w, s: ops.w4a16_gemm(x, torch.zeros(8, 32, dtype=torch.int32), s.half().view(8, 1).expand(8, 2).contiguous(),
                                   None, 128, None),
    lambda x, w, s: ops.w8a8_gemm(x.to(torch.int8), torch.ones(64), w, s, None, torch.float16),
    lambda x, w, s: ops.w8a8_linear(x, w, s, None, torch.float16, False),
    lambda x, w, s: ops.w8a8_linear_fake(x, w, s, None),
])
def test_workspace_is_asked_under_the_device_guard(monkeypatch, call):
    lib = _Library()

    @contextlib.contextmanager
    def guard(t):
        lib.device = "the tensor's"
        yield
        lib.device = "current"

    monkeypatch.setattr(ops, "_need", lambda *a, **k: None)
    monkeypatch.setattr(ops, "_dev", guard)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops._lib, "load", lambda: lib)
    call(torch.randn(64, 256).half(), torch.zeros(8, 256, dtype=torch.int8), torch.ones(8))
    assert lib.launched and lib.asked and {d for _, d in lib.asked + lib.launched} == {"the tensor's"}

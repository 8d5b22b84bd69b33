"""How many key ranges the attention entry points of the hybrid decoders ask their kernels for.  No GPU: the library call is recorded."""
from __future__ import annotations

import pytest
import torch


class _Recorder:
    """Stands in for the kernel library: remembers the `splits` argument of the last launch, hands other calls on."""

    def __init__(self, real):
        self.real, self.splits = real, None

    def __getattr__(self, name):
        def launch(*a):
            self.splits = a[-3]  # splits, workspace, stream end every signature
            return 0

        return launch if name.endswith("_attn") else getattr(self.real, name)


@pytest.fixture
def launched(monkeypatch):
    from mini_sglang_amd import _lib, mixops

    rec = _Recorder(_lib.mix_lib())
    monkeypatch.setattr(mixops, "mix_lib", lambda: rec)
    monkeypatch.setattr(mixops, "_dev", lambda *a: None)
    monkeypatch.setattr(mixops, "_stream", lambda: None)
    return rec


def _i32(*x):
    return torch.tensor(x, dtype=torch.int32)


def _window(rec, T, batch, width, dtype=torch.bfloat16, H=16, G=4, d=128, window=0, **kw):
    from mini_sglang_amd import mixops

    z = lambda *s: torch.zeros(s, dtype=dtype)  # noqa: E731
    rec.splits = None
    mixops.window_attn(z(T, H * d), z(T, H * d + H), H * d, z(8, G * d), z(8, G * d), torch.zeros((max(batch, 1), width), dtype=torch.int32), _i32(*range(batch)),
                       _i32(*[1] * batch), _i32(*range(batch + 1)), batch, H, G, d, d, window, 0.1, torch.eye(H), **kw)
    return rec.splits


def test_window_without_requests(launched):
    """A step without requests has no groups to divide by."""
    assert _window(launched, 0, 0, 4096) == 1

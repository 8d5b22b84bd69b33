"""Which batches share what a backend keeps for its decode steps: host-side rules, without a GPU."""
from types import SimpleNamespace

import pytest
import torch


@pytest.fixture
def backend(monkeypatch):
    """A backend of 16 query heads on 8 whose kernels are not called, on a device of 256 compute units."""
    from mini_sglang_amd import attention

    b = object.__new__(attention.HipAttnBackend)
    b.qo_heads, b.kv_heads, b.head_dim, b._small_heads = 16, 8, 128, 64
    monkeypatch.setattr(attention._lib, "lib", lambda: SimpleNamespace(msgl_device_cu_count=lambda: 256))
    monkeypatch.setattr(attention.ops, "decode_layers_supported", lambda *a: True)
    return b


def _batch(phase, n=3):
    from mini_sglang_amd.attention import HipAttnMetadata

    v = torch.zeros(n, dtype=torch.int32)
    md = HipAttnMetadata(cu_seqlens_q=torch.arange(n + 1, dtype=torch.int32), seq_lens=v + 9, req_rows=v, batch=n, max_seqlen_q=1, max_seqlen_k=9)
    return SimpleNamespace(phase=phase, positions=v, out_loc=v, attn_metadata=md)


def test_one_token_prompts_take_no_part_in_the_decode_steps_launch(backend):
    """A prompt whose requests all extend by one token (a full hit of the prefix cache, a remainder of one token) may run beside a decode step on another
    stream, and that step's launch has its workgroups meet in memory that the backend has once."""
    assert backend.takes_layers(_batch("decode"), 1024, 3072)
    assert not backend.takes_layers(_batch("prefill"), 1024, 3072)

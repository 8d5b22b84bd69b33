"""Which batches share what a backend keeps for its decode steps: host-side rules, without a GPU."""
from types import SimpleNamespace

import pytest
import torch


@pytest.fixture
def backend(monkeypatch):
    """A backend of 16 query heads on 8 whose kernels are not called, on a device of 256 compute units."""
    from mini_sglang_amd import attention

    b = object.__new__(attention.HipAttnBackend)
    b.qo_heads, b.kv_heads, b.head_dim, b._small_heads, b.device = 16, 8, 128, 64, torch.device("cpu")
    b._layers_workspaces, b.ctx = {}, SimpleNamespace(page_table=torch.zeros(4, 32, dtype=torch.int32))
    monkeypatch.setattr(attention._lib, "lib", lambda: SimpleNamespace(msgl_device_cu_count=lambda: 256))
    monkeypatch.setattr(attention.ops, "decode_layers_supported", lambda *a: True)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    return b


def _batch(phase, n=3):
    from mini_sglang_amd.attention import HipAttnMetadata

    v = torch.zeros(n, dtype=torch.int32)
    md = HipAttnMetadata(cu_seqlens_q=torch.arange(n + 1, dtype=torch.int32), seq_lens=v + 9, req_rows=v, batch=n, max_seqlen_q=1, max_seqlen_k=9)
    return SimpleNamespace(phase=phase, positions=v, out_loc=v, attn_metadata=md)


def test_one_token_prompts_take_no_part_in_the_decode_steps_launch(backend):
    """A prompt whose requests all extend by one token (a full hit of the prefix cache, a remainder of one token) may run beside a decode step on another
    stream, and that step's launch has its workgroups meet in memory that the backend has once."""
    assert backend.takes_layers(_batch("decode"), 1024, 3072, 28)
    assert not backend.takes_layers(_batch("prefill"), 1024, 3072, 28)


def test_the_first_step_of_a_model_is_not_captured_as_one_launch(backend, monkeypatch):
    """The launch's workgroups start from zeros that are written once, eagerly: a capture in front of every step takes the separate launches, one after a
    step of the same model does not; models of other sizes have memory of their own."""
    from mini_sglang_amd import attention

    monkeypatch.setattr(attention.ops, "decode_layers_workspace_bytes", lambda b, layers, hidden, hq, hkv, inter: b * layers * (hidden + inter))
    capturing = [True]
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    assert not backend.takes_layers(_batch("decode"), 1024, 3072, 28)
    capturing[0] = False
    assert backend.takes_layers(_batch("decode"), 1024, 3072, 28)
    first = backend._layers_workspace(28, 1024, 3072)
    assert first.numel() == 8 * 28 * 4096 and not first.any()
    capturing[0] = True
    assert backend.takes_layers(_batch("decode"), 1024, 3072, 28) and backend._layers_workspace(28, 1024, 3072) is first
    assert not backend.takes_layers(_batch("decode"), 1024, 3072, 40)
    capturing[0] = False
    assert backend._layers_workspace(40, 1024, 3072).numel() == 8 * 40 * 4096 and backend._layers_workspace(28, 1024, 3072) is first


def test_the_error_word_is_not_asked_for_inside_a_capture(backend, monkeypatch):
    """Every 64th batch's metadata asks for the one-launch steps' error word: a copy and an event, which have no place in somebody's graph."""
    polls, capturing = [], [False]
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    monkeypatch.setattr(type(backend), "poll_errors", lambda self: polls.append(1))
    backend.tp_size, backend._md_calls, backend._layers_workspaces = 1, 0, {(28, 1024, 3072): torch.zeros(1)}
    batch = SimpleNamespace(padded_reqs=None)  # (what follows is not looked at)
    for i in range(4 * 64):
        capturing[0] = i >= 2 * 64
        with pytest.raises(TypeError):
            backend.prepare_metadata(batch)
    assert len(polls) == 2


@pytest.mark.parametrize("hidden,heads,kv_heads,width,most", [(1024, 16, 8, 4096, 8), (1024, 16, 8, 40960, 4), (768, 16, 8, 4096, 8), (512, 8, 8, 4096, 0),
                                                              (1024, 16, 4, 4096, 4), (768, 24, 4, 4128, 0), (1024, 6, 3, 64, 4), (1024, 16, 2, 4096, 3),
                                                              (1024, 8, 1, 4096, 3), (1024, 8, 1, 8192, 0), (512, 8, 1, 4096, 0)])
def test_where_one_launch_is_ahead(backend, hidden, heads, kv_heads, width, most):
    """Steps take the one launch only where it was measured ahead at every length that the engine's page table admits: up to `most` requests."""
    from mini_sglang_amd.attention import SMALL_DECODE_HEADS

    backend.qo_heads, backend.kv_heads, backend.ctx.page_table = heads, kv_heads, torch.zeros(2, width, dtype=torch.int32)
    backend._small_heads = SMALL_DECODE_HEADS * (2 if kv_heads <= 2 or width <= 4096 else 1)
    assert [n for n in range(1, 9) if backend.takes_layers(_batch("decode", n), hidden, 3072, 28)] == list(range(1, most + 1))


@pytest.mark.parametrize("small", [True, False], ids=["small batch", "planned"])
def test_one_token_prompts_have_partial_sums_of_their_own(backend, monkeypatch, small):
    """Decode steps share the backend's scratch; a one-token prompt keeps its own with its batch, the same for all its layers."""
    from mini_sglang_amd import attention

    seen = []
    if small:
        monkeypatch.setattr(attention.ops, "attn_decode_small_ranges", lambda *a: 1)
        monkeypatch.setattr(attention.ops, "attn_decode_small", lambda *a, **k: seen.append(a[10]))
    else:
        backend._small_heads = 0
        monkeypatch.setattr(attention.ops, "attn_decode", lambda *a, **k: seen.append(a[8]))
    pool = torch.zeros(16, 8, 128)
    backend.scale, backend.max_bs, backend.capacity, backend.slot_run, backend.device = 1.0, 4, 64, 1, torch.device("cpu")
    backend._cap_plan = None
    backend.kvcache = SimpleNamespace(k_cache=lambda i: pool, v_cache=lambda i: pool, store_kv=lambda *a: None, dtype=torch.float32)
    backend._workspace = torch.empty(4096, dtype=torch.uint8)
    q, k = torch.zeros(3, 16, 128), torch.zeros(3, 8, 128)
    for phase in ("decode", "prefill", "prefill"):
        batch = _batch(phase)
        batch.attn_metadata.plan = torch.zeros(1, dtype=torch.int32)
        for layer in range(2):
            backend.forward(q, k, k, layer, batch)
    assert len(seen) == 6 and seen[0] is seen[1] is backend._workspace
    assert seen[2] is seen[3] and seen[4] is seen[5] and len({id(t) for t in seen}) == 3
    assert seen[2].numel() == backend._workspace.numel()

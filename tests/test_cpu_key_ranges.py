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


def _latent(rec, T, batch, width, H=16, **kw):
    from mini_sglang_amd import mixops

    mixops.latent_attn(torch.zeros(T, H, 512), torch.zeros(T, H, 576), torch.zeros(8, 576, dtype=torch.bfloat16), torch.zeros((batch, width), dtype=torch.int32),
                       _i32(*range(batch)), _i32(*[1] * batch), _i32(*range(batch + 1)), batch, 512, 0.1, **kw)
    return rec.splits


def _diff(rec, T, batch, width, H=16, G=4, window=0, keep=0, **kw):
    from mini_sglang_amd import mixops

    z = lambda *s: torch.zeros(s, dtype=torch.bfloat16)  # noqa: E731
    mixops.diff_attn(z(T, H * 128), torch.zeros(T, H * 128), z(8, G * 128), z(8, G * 128), torch.zeros((batch, width), dtype=torch.int32), _i32(*range(batch)),
                     _i32(*[1] * batch), _i32(*range(batch + 1)), batch, H, G, 64, 128, 0.1, window, keep, torch.ones(1), 0.5, 1e-5, **kw)
    return rec.splits


@pytest.mark.parametrize("call", [_latent, _window, _diff], ids=["latent", "window", "maps"])
def test_ranges_follow_the_longest_sequence_not_the_table(launched, call):
    """An engine's table is as wide as the longest sequence it allows: the batch's longest one decides, the width only where it is not given."""
    wide = 40960
    assert call(launched, 100, 1, wide, max_keys=100) == 1  # a short fresh portion: one range
    for n in (100, 300, 500, 1000, 5000):
        assert call(launched, 20, 1, wide, max_keys=n) == call(launched, 20, 1, n), n
    assert call(launched, 20, 1, wide, max_keys=5000) == call(launched, 20, 1, wide) == 8
    assert call(launched, 20, 1, wide, max_keys=100, splits=3) == 3  # the caller's own number stays
    assert call(launched, 8192, 4, wide, max_keys=4000) == 1  # groups enough


def test_ranges_stay_inside_the_window(launched):
    assert _window(launched, 20, 1, 40960, window=256, max_keys=9000) == 2
    assert _diff(launched, 20, 1, 40960, window=64, keep=64, max_keys=9000) == 1
    assert _diff(launched, 20, 1, 40960, window=1024, keep=64, max_keys=9000) == 4


def test_window_ranges_of_the_plain_kernel(launched):
    """fp32 engines and head counts that the matrix cores do not take: a range from 64 keys on."""
    for kw in ({"dtype": torch.float32}, {"H": 12}, {"G": 8}, {"d": 136}):
        assert _window(launched, 20, 1, 40960, max_keys=64, **kw) == 1 and _window(launched, 20, 1, 40960, max_keys=100, **kw) == 2
        assert _window(launched, 20, 1, 40960, max_keys=5000, **kw) == 8


def test_delta_rule_blocks_where_they_are_faster():
    """Portions on both sides of the line between the token loop and blocks of 16 tokens, the measured one at each; a longest portion that the
    caller names decides over the mean."""
    from mini_sglang_amd.mixops import delta_in_blocks

    for batch, each, H, d, channel, want in [
            (1, 5, 16, 128, False, False), (1, 6, 16, 128, False, True), (8, 6, 16, 128, True, True), (16, 6, 16, 128, False, False), (16, 8, 16, 128, False, True),
            (64, 6, 4, 128, True, True), (1, 9, 16, 64, False, False), (1, 10, 16, 64, False, True), (40, 16, 16, 64, False, False), (16, 28, 16, 64, False, True),
            (1, 5, 8, 64, True, False), (4, 6, 8, 64, True, True), (16, 8, 16, 64, True, False), (64, 13, 16, 64, True, True), (32, 1, 16, 128, True, False)]:
        assert delta_in_blocks(batch, batch * each, H, d, channel, longest=each) == want, (batch, each, H, d, channel)
    assert delta_in_blocks(40, 640, 16, 64, False)  # many requests that may hide a long portion
    assert delta_in_blocks(16, 95, 16, 128, False, longest=80) and not delta_in_blocks(16, 95, 16, 128, False)
    assert not delta_in_blocks(64, 384, 16, 128, False, longest=6) and not delta_in_blocks(64, 64, 16, 64, True, longest=1)


def test_delta_rule_pieces_where_the_token_loop_takes_long_portions(monkeypatch):
    """The list of a long portion's pieces is built for head sizes that have no form in blocks, and for no other: they read none at that length."""
    from types import SimpleNamespace as N

    from mini_sglang_amd import attention, mixops

    empty = torch.empty
    monkeypatch.setattr(attention.torch, "empty", lambda *a, pin_memory=False, **kw: empty(*a, **kw))
    ctx = N(kv_cache=N(device=torch.device("cpu")), page_table=torch.zeros((4, 2048), dtype=torch.int32))
    n = 2 * attention.MixAttnBackend.DELTA_CHUNK
    for dim, vdim, kind, want in [(128, 128, "delta", False), (64, 96, "channel_delta", False), (64, 80, "delta", True), (96, 96, "channel_delta", True)]:
        layer = N(kind=kind, dim=dim, vdim=vdim)
        for layers in ([layer], [N(kind="parallel", left=N(kind="window"), right=layer)]):
            batch = N(padded_reqs=[N(extend_len=k, device_len=k + 5, table_idx=i) for i, k in enumerate((1, n, 7))])
            attention.MixAttnBackend(N(layers=layers), ctx).prepare_metadata(batch)
            md = batch.attn_metadata
            assert (md.delta_chunks is not None) == want and (want or mixops.delta_in_blocks(3, n + 8, 16, dim, kind == "channel_delta", md.max_seqlen_q))
            if want:
                items, first, count = md.delta_chunks
                assert count == 4 and items.view(-1, 3).tolist() == [[0, 0, 1], [1, 0, n // 2], [1, n // 2, n], [2, 0, 7]] and first.tolist() == [0, 1, 3, 4]


def test_prefill_heads_go_in_pairs_by_length_of_chains():
    """Two heads a workgroup: the rule's both bands, their lines in number of chains, mean length, longest one and group."""
    import numpy as np

    from mini_sglang_amd import ops

    def pairs(hq, hkv, *portions):  # portions: (requests, new tokens, tokens before them)
        q = np.array([n for c, n, _ in portions for _ in range(c)], dtype=np.int64)
        k = np.array([n + o for c, n, o in portions for _ in range(c)], dtype=np.int64)
        return ops.prefill_pairs(int(((q + 127) // 128).sum()), hq, hkv, q, k)

    # from 3072 chains on, 36 tiles on average
    assert pairs(64, 8, (1, 8192, 16384)) and pairs(64, 8, (1, 6144, 0)) and pairs(32, 16, (3, 4300, 2000)) and pairs(8, 1, (12, 4096, 1000))
    assert not pairs(64, 8, (1, 6016, 9000))                                                   # 3008 chains
    assert not pairs(128, 8, (8, 1910, 0)) and not pairs(64, 8, (4, 2030, 500)) and not pairs(24, 4, (42, 340, 1000))  # 16 - 24 tiles
    assert not pairs(40, 8, (1, 16384, 8192)) and not pairs(12, 4, (1, 65536, 0))              # odd groups
    # two rounds nearly full, 15 tiles on average, none much longer than an even share
    assert pairs(64, 8, (1, 2048, 0)) and pairs(64, 8, (1, 1792, 0)) and pairs(8, 1, (9, 1700, 6000)) and pairs(16, 8, (3, 2400, 0))
    assert not pairs(64, 8, (1, 2176, 0)) and not pairs(64, 8, (1, 1664, 0))                   # 1088, 832 chains
    assert not pairs(24, 4, (5, 1000, 0))                                                      # 8 tiles
    assert not pairs(8, 1, (1, 6784, 0), (3, 2500, 0)) and pairs(8, 1, (4, 3600, 0))           # one chain of 106 tiles, even ones

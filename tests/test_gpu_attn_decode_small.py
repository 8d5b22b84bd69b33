"""msgl_attn_decode_small: qk-norm, RoPE, K / V store and decode attention of a small batch against the separate row kernel (stored
rows: the same bits) and attention in float64."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops(dev):
    from mini_sglang_amd import ops as o

    return o


def _case(ops, dev, dtype, hq, hkv, lens, page, norm, rope, ranges=None, seed=0):
    from mini_sglang_amd import flashinfer_compat as fi

    g = torch.Generator(device=dev).manual_seed(seed)
    rnd = lambda *s: torch.randn(s, generator=g, device=dev).to(dtype)  # noqa: E731
    B, need = len(lens), [-(-n // page) for n in lens]
    order = torch.randperm(sum(need), generator=torch.Generator().manual_seed(seed)).to(dev)
    table = torch.zeros((B + 2, (max(lens) + 31) // 32 * 32), dtype=torch.int32, device=dev)
    rows = torch.randperm(B + 2, generator=torch.Generator().manual_seed(seed + 1))[:B].to(torch.int32).to(dev)
    at, slots = 0, []
    for r, n, c in zip(rows.tolist(), lens, need):
        s = (order[at: at + c, None] * page + torch.arange(page, device=dev)).reshape(-1)[:n]
        table[r, :n] = s.int()
        slots.append(s)
        at += c
    pool = sum(need) * page
    kc, vc = rnd(pool, hkv, 128), rnd(pool, hkv, 128)
    loc = torch.stack([s[-1] for s in slots]).int()
    # what lies in the new slots and in slots of no request must not be read into a result
    used = torch.zeros(pool, dtype=torch.bool, device=dev)
    for s in slots:
        used[s[:-1]] = True
    kc[~used] = math.nan
    vc[~used] = math.nan
    qkv = rnd(B, (hq + 2 * hkv) * 128 + 8)[:, : (hq + 2 * hkv) * 128]
    q, k, v = qkv.split([hq * 128, hkv * 128, hkv * 128], dim=1)
    seq = torch.tensor(lens, dtype=torch.int32, device=dev)
    pos = seq - 1
    qw, kw = (rnd(128), rnd(128)) if norm else (None, None)
    cs = fi.build_cos_sin_cache(128, max(lens) + 1, 1e4, None, device=dev) if rope else None
    # the separate row kernel on copies (a rotation by nothing where there is none)
    one = torch.cat([torch.ones(64, device=dev), torch.zeros(64, device=dev)]).repeat(max(lens) + 1, 1).contiguous()
    q1, k1, v1, kc1, vc1 = q.clone(), k.clone(), v.clone(), kc.clone(), vc.clone()
    ops.qk_norm_rope_store(q1, k1, v1, qw, kw, 1e-6, pos, cs if rope else one, kc1.view(pool, -1), vc1.view(pool, -1), loc, 128)
    R = ranges or ops.attn_decode_small_ranges(B, hkv, table.shape[1])
    ws = torch.empty(B * R * hq * 130, dtype=torch.float32, device=dev)
    out = torch.full((B + 1, hq * 128 + 8), 7.0, dtype=dtype, device=dev)
    before = qkv.clone()

    def launch():
        ops.attn_decode_small(out[:B, : hq * 128], q, k, v, kc, vc, loc, table, rows, seq, ws, R, 128 ** -0.5, qw, kw, 1e-6,
                              pos if rope else None, cs)

    launch()
    idx = loc.long()
    assert torch.equal(kc[idx], kc1[idx]) and torch.equal(vc[idx], vc1[idx])
    rest = torch.ones(pool, dtype=torch.bool, device=dev)
    rest[idx] = False
    assert torch.equal(kc[rest].view(torch.int16), kc1[rest].view(torch.int16)) and torch.equal(vc[rest].view(torch.int16), vc1[rest].view(torch.int16))
    assert torch.equal(qkv, before) and bool((out[B:] == 7).all()) and bool((out[:, hq * 128:] == 7).all())
    G, eps = hq // hkv, torch.finfo(dtype).eps
    for b, s in enumerate(slots):
        kk, vv, qq = kc1[s].double(), vc1[s].double(), q1[b].view(hq, 128).double()
        for h in range(hq):
            sc = (kk[:, h // G] @ qq[h]) * 128 ** -0.5
            p = torch.softmax(sc, dim=0)
            want = p @ vv[:, h // G]
            got = out[b, h * 128: (h + 1) * 128].double()
            # weights and result rounded to the 16-bit type (their sum is not), scores from fp32 sums of 128 products
            fp32 = 2.0 ** -22 * 128 * (kk[:, h // G].abs() @ qq[h].abs()).max() * 128 ** -0.5
            bound = (eps / 2 + 2 * fp32 + 1e-5) * (p @ vv[:, h // G].abs()) + eps / 2 * want.abs() + 1e-7
            assert bool(((got - want).abs() <= bound).all()), (b, h, (got - want).abs().max())
    first = out.clone()
    launch()  # again over the rows that it stored
    assert torch.equal(out, first)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("hq,hkv", [(1, 1), (4, 2), (5, 1), (16, 8), (8, 1), (21, 3)])
@pytest.mark.parametrize("lens,page", [([1], 1), ([15, 16, 17], 16), ([127, 128, 129, 130], 1), ([2049, 1, 300], 256)])
def test_small_decode_is_row_kernel_and_attention(ops, dev, dtype, hq, hkv, lens, page):
    _case(ops, dev, dtype, hq, hkv, lens, page, norm=True, rope=True)


@pytest.mark.parametrize("norm,rope", [(False, True), (True, False), (False, False)])
def test_small_decode_without_norm_or_rotation(ops, dev, norm, rope):
    _case(ops, dev, torch.bfloat16, 8, 2, [40, 700], 16, norm, rope)


@pytest.mark.parametrize("ranges", [1, 2, 5, 63, 64])
def test_small_decode_over_numbers_of_ranges(ops, dev, ranges):
    """One range finishes in the kernel; more ranges than a request has pieces; several tiles per wave."""
    _case(ops, dev, torch.bfloat16, 6, 2, [4000, 9, 513], 16, True, True, ranges=ranges)


def test_small_decode_refusals(ops, dev):
    x = torch.zeros((1, 9 * 128), dtype=torch.bfloat16, device=dev)
    kv, pool = torch.zeros((1, 128), dtype=torch.bfloat16, device=dev), torch.zeros((4, 1, 128), dtype=torch.bfloat16, device=dev)
    i32 = torch.ones(32, dtype=torch.int32, device=dev)
    for q, ranges, floats in ((x, 1, 9 * 130), (x[:, :128], 65, 65 * 130), (x[:, :128], 2, 130)):  # 9 heads per kv head; ranges; workspace
        with pytest.raises(Exception):
            ops.attn_decode_small(torch.empty_like(q), q, kv, kv, pool, pool.clone(), i32, i32.view(1, 32), None, i32,
                                  torch.empty(floats, dtype=torch.float32, device=dev), ranges, 1.0)


@pytest.mark.parametrize("hq,hkv,d,width,most", [(16, 8, 128, 4096, 8), (16, 8, 128, 4128, 4), (40, 8, 128, 40960, 4), (10, 2, 128, 40960, 32), (5, 1, 128, 40960, 64),
                                                 (32, 32, 128, 40960, 1), (18, 2, 128, 512, 0), (16, 8, 64, 512, 0)])
def test_batches_that_take_the_small_kernel(dev, hq, hkv, d, width, most):
    """The rule by requests x kv heads on both sides of its lines: a table of up to 4096 tokens, one or two kv heads, other heads than the kernel's."""
    from types import SimpleNamespace

    from mini_sglang_amd.attention import HipAttnBackend
    from mini_sglang_amd.core import Context
    from mini_sglang_amd.kvcache import create_kvcache_pool
    from mini_sglang_amd.model import ModelConfig

    m = ModelConfig(num_layers=1, num_qo_heads=hq, num_kv_heads=hkv, head_dim=d, hidden_size=256, vocab_size=64, intermediate_size=64)
    ctx = Context(16)
    ctx.page_table = torch.zeros((80, width), dtype=torch.int32, device=dev)
    ctx.kv_cache = create_kvcache_pool(m, 2, 16, torch.bfloat16, dev)
    backend = HipAttnBackend(m, ctx)
    says = [b for b in range(1, 80) if backend.small_decode(SimpleNamespace(attn_metadata=SimpleNamespace(max_seqlen_q=1, batch=b)))]
    assert says == list(range(1, most + 1))
    assert not backend.small_decode(SimpleNamespace(attn_metadata=SimpleNamespace(max_seqlen_q=2, batch=1)))


def test_replayed_batches_of_both_kernels_keep_their_plan(dev, monkeypatch):
    """An engine whose captured batch sizes lie on both sides of the rule: replays of either after the other, against eager runs."""
    from mini_sglang_amd import ops
    from mini_sglang_amd.core import SamplingParams
    from mini_sglang_amd.engine import Engine, EngineConfig
    from mini_sglang_amd.model import ModelConfig
    from mini_sglang_amd.offline import OfflineRunner
    from replay_util import record_offline_runner, replay_forward

    m = ModelConfig(2, 16, 8, 128, 1024, 512, 1024, name="small")
    cfg = EngineConfig(model=m, dtype=torch.bfloat16, max_running_req=16, page_size=16, cuda_graph_bs=[2, 4, 16], max_seq_len_override=8192,
                       num_page_override=600, seed=5, gemm_tune="off")
    eng = Engine(cfg, dev)
    try:
        assert eng.attn_backend._cap_planned == {16}
        rec = []
        runner = OfflineRunner(eng, max_extend_tokens=4096, seed=1)
        record_offline_runner(runner, eng, rec)
        for n in (16, 3, 16, 2):
            prompts = [[(7 * i + j) % 500 for j in range(5 + 37 * i)] for i in range(n)]
            runner.generate(prompts, [SamplingParams(temperature=0.0, max_tokens=3, ignore_eos=True) for _ in prompts])
        decodes = [f for f in rec if f["phase"] == "decode"]
        assert {f["size"] for f in decodes} == {16, 3, 2} and all(f["graph"] for f in decodes)
        last = decodes[-1]  # its pages are still what they were
        a = replay_forward(eng, last).float().cpu()
        monkeypatch.setattr(eng.graph_runner, "can_use_cuda_graph", lambda batch: False)
        b = replay_forward(eng, dict(last, graph=False)).float().cpu()
        assert torch.equal(a, b) and torch.equal(a, last["logits"])
    finally:
        eng.shutdown()
        ops.reset_gemm_plans()

"""GPU parity: paged varlen causal prefill attention (MFMA) vs the CPU oracle.

Covers the three metadata regimes of P/attention/fa.py:84-90: no cache hit (q_len == k_len),
partial radix hit / chunked prefill (q_len < k_len, bottom-right aligned mask), and mixed
batches with ragged lengths around the 128-row / 64-key tile edges.
"""
import math

import pytest
import torch

from oracle import ref_ops

pytestmark = pytest.mark.gpu

TOL = dict(atol=8e-3, rtol=2 ** -6)  # P is rounded to bf16 before P.V (as FA-style kernels do)


@pytest.fixture(scope="module")
def ops(dev):
    from mini_sglang_amd import ops as _ops

    return _ops


def build(g, specs, hq, hkv, page_size, dtype=torch.bfloat16):
    """specs: list of (cached_len, device_len) per request."""
    D = 128
    B = len(specs)
    max_seq = (max(dl for _, dl in specs) + 31) // 32 * 32
    pages_per = (max_seq + page_size - 1) // page_size
    n_pages = (B + 2) * pages_per + 2
    slots = n_pages * page_size
    k = torch.randn((slots, hkv, D), generator=g).to(dtype)
    v = torch.randn((slots, hkv, D), generator=g).to(dtype)
    poison = (n_pages - 1) * page_size
    k[poison:] = float("nan")
    v[poison:] = float("nan")
    perm = torch.randperm(n_pages - 2, generator=g)
    table = torch.full((B + 2, max_seq), poison, dtype=torch.int32)
    rows = torch.randperm(B + 2, generator=g)[:B].tolist()
    pp = 0
    for (cl, dl), row in zip(specs, rows):
        need = (dl + page_size - 1) // page_size
        pg = perm[pp: pp + need].to(torch.int32) * page_size
        pp += need
        tok = (pg.unsqueeze(1) + torch.arange(page_size, dtype=torch.int32)).flatten()
        table[row, :dl] = tok[:dl]
    q_lens = [dl - cl for cl, dl in specs]
    T = sum(q_lens)
    qkv = torch.randn((T, (hq + 2 * hkv) * D), generator=g).to(dtype)
    return dict(k=k, v=v, table=table, rows=rows, q_lens=q_lens, k_lens=[dl for _, dl in specs], qkv=qkv, hq=hq,
                hkv=hkv)


@pytest.fixture(params=[0, 2], ids=["default_dma", "tr_read"])
def impl(request):
    """Both kernels (include/msgl_hip.h: 0 = the default = impl 4, DMA-staged; 2 = its register-staged predecessor, the A/B
    partner)."""
    return request.param


def run(ops, dev, c, impl=0, order="heavy"):
    import numpy as np

    from mini_sglang_amd.attention import prefill_tile_order

    D, hq = 128, c["hq"]
    qkv = c["qkv"].to(dev)
    T = qkv.shape[0]
    q = qkv[:, : hq * D].view(T, hq, D)
    out = torch.zeros((T, hq, D), dtype=qkv.dtype, device=dev)
    cu_q = torch.tensor([0] + c["q_lens"], dtype=torch.int32).cumsum(0).to(torch.int32)
    qt = ops.prefill_q_tile(impl)  # rows per q tile of the kernel (128)
    tiles = [(n + qt - 1) // qt for n in c["q_lens"]]
    tile_cu = torch.tensor([0] + tiles, dtype=torch.int32).cumsum(0).to(torch.int32)
    tile_order = None
    if order == "heavy":
        tile_order = torch.from_numpy(prefill_tile_order(np.array(c["q_lens"], dtype=np.int64),
                                                         np.array(c["k_lens"], dtype=np.int64),
                                                         np.array(tiles, dtype=np.int64), qt)).to(dev)
    elif order == "reversed":
        tile_order = torch.arange(int(tile_cu[-1]) - 1, -1, -1, dtype=torch.int32, device=dev)
    ops.attn_prefill(out, q, c["k"].to(dev), c["v"].to(dev), c["table"].to(dev),
                     torch.tensor(c["rows"], dtype=torch.int32, device=dev),
                     torch.tensor(c["k_lens"], dtype=torch.int32, device=dev), cu_q.to(dev), tile_cu.to(dev),
                     len(c["q_lens"]), int(tile_cu[-1]), D ** -0.5, tile_order=tile_order, impl=impl)
    torch.cuda.synchronize()
    return out.cpu()


def oracle(c):
    D, hq = 128, c["hq"]
    T = c["qkv"].shape[0]
    q = c["qkv"][:, : hq * D].reshape(T, hq, D)
    return ref_ops.paged_attention_ref(q, c["k"], c["v"], c["table"], c["rows"], c["k_lens"], c["q_lens"],
                                       D ** -0.5, double=True)


@pytest.mark.parametrize("hq,hkv", [(16, 8), (40, 8), (8, 1), (4, 4)])
@pytest.mark.parametrize("page_size", [1, 16])
def test_prefill_no_cache_hit(ops, dev, impl, hq, hkv, page_size):
    g = torch.Generator().manual_seed(hq + page_size)
    specs = [(0, n) for n in (1, 5, 31, 32, 33, 63, 64, 65, 127, 128, 129, 300, 517)]
    c = build(g, specs, hq, hkv, page_size)
    out = run(ops, dev, c, impl)
    assert torch.isfinite(out.float()).all()
    torch.testing.assert_close(out.double(), oracle(c), **TOL)


def test_prefill_partial_hit_and_chunked(ops, dev, impl):
    """q_len < k_len: radix prefix hits (page-aligned cached_len) and chunked-prefill continuation."""
    g = torch.Generator().manual_seed(1)
    specs = [(16, 40), (64, 65), (128, 400), (1000, 1001), (512, 1024), (0, 7), (256, 257 + 128), (48, 49)]
    c = build(g, specs, 40, 8, 16)
    out = run(ops, dev, c, impl)
    torch.testing.assert_close(out.double(), oracle(c), **TOL)


def test_prefill_tile_order_does_not_change_results(ops, dev):
    """tile_order is a scheduling hint: natural, heaviest-first and reversed orders are bit-identical."""
    g = torch.Generator().manual_seed(11)
    specs = [(0, 300), (128, 400), (0, 1), (512, 1024), (0, 129)]
    c = build(g, specs, 10, 2, 16)
    for impl in (0, 2):
        a = run(ops, dev, c, impl, order="heavy")
        assert torch.equal(a, run(ops, dev, c, impl, order=None))
        assert torch.equal(a, run(ops, dev, c, impl, order="reversed"))
        torch.testing.assert_close(a.double(), oracle(c), **TOL)


def test_prefill_generations_agree(ops, dev):
    """Same fragment ownership and accumulation order in both kernels => identical bits."""
    g = torch.Generator().manual_seed(12)
    c = build(g, [(0, 517), (64, 200), (1000, 1100)], 16, 8, 1)
    # the DMA-staged kernel (4, the default) keeps the register-staged kernel's (2) math, fragment ownership and accumulation
    # order per query row: identical bits, also on a batch with cache hits, a ragged tail, a request shorter than one tile
    # and one spanning several tiles
    for cc in (c, build(torch.Generator().manual_seed(13), [(0, 1), (0, 255), (0, 257), (300, 1100), (0, 700), (4096, 4200)], 10, 2, 16)):
        a = run(ops, dev, cc, 2)
        assert torch.equal(a, run(ops, dev, cc, 4))
        assert torch.equal(a, run(ops, dev, cc, 0))


def test_prefill_rejects_removed_and_diagnostic_impl_codes(ops, dev):
    """a stray MSGL_PREFILL_IMPL / impl argument must not select a timing-only ablation kernel (wrong results)
    or a removed generation: production builds accept 0, 2, 4 only."""
    from mini_sglang_amd._lib import MsglError

    c = build(torch.Generator().manual_seed(14), [(0, 40)], 4, 2, 16)
    for bad in (1, 3, 5, 16, 17, 64, 65, 128, 511, -1):
        with pytest.raises(MsglError):
            run(ops, dev, c, bad)


def test_prefill_long(ops, dev, impl):
    g = torch.Generator().manual_seed(2)
    specs = [(0, 2048), (1024, 3000)]
    c = build(g, specs, 16, 8, 1)
    out = run(ops, dev, c, impl)
    torch.testing.assert_close(out.double(), oracle(c), **TOL)


def test_prefill_fp16(ops, dev, impl):
    g = torch.Generator().manual_seed(3)
    c = build(g, [(0, 200), (32, 90)], 16, 8, 1, dtype=torch.float16)
    out = run(ops, dev, c, impl)
    torch.testing.assert_close(out.double(), oracle(c), atol=2e-3, rtol=2 ** -8)


def test_prefill_transpose_detecting(ops, dev, impl):
    """Asymmetric structured inputs (guide rule 16): V[key, d] = key + d/1000 with uniform
    attention => O[q, d] = mean_key(key) + d/1000; a swapped row/col layout cannot pass."""
    g = torch.Generator().manual_seed(4)
    c = build(g, [(0, 96)], 8, 8, 1)
    D = 128
    slots = c["table"][c["rows"][0], :96].long()
    c["k"][slots] = 0
    keys = torch.arange(96, dtype=torch.float32).view(96, 1, 1) / 16.0
    dd = torch.arange(D, dtype=torch.float32).view(1, 1, D) / 64.0
    hh = torch.arange(8, dtype=torch.float32).view(1, 8, 1)
    c["v"][slots] = (keys + dd + hh).to(torch.bfloat16)
    out = run(ops, dev, c, impl)
    torch.testing.assert_close(out.double(), oracle(c), **TOL)


def test_prefill_matches_decode_on_last_token(ops, dev):
    """The last query row of a prefill equals a decode step over the same KV."""
    import test_gpu_attn_decode as td

    g = torch.Generator().manual_seed(5)
    c = build(g, [(0, 333), (100, 777)], 40, 8, 1)
    out = run(ops, dev, c)
    D, hq = 128, 40
    last = [c["q_lens"][0] - 1, sum(c["q_lens"]) - 1]
    case = dict(k=c["k"], v=c["v"], table=c["table"], rows=c["rows"], lens=c["k_lens"],
                qkv=c["qkv"][last].contiguous(), hq=hq, hkv=8, D=D)
    dec, _ = td.run_decode(ops, dev, case)
    torch.testing.assert_close(out[last].float(), dec.float(), atol=8e-3, rtol=2 ** -6)


def test_prefill_row_sum_of_unrounded_weights(ops, dev, impl):
    """A row's sum takes the fp32 weights, the products the bf16 ones: all weights but one are 0.25062, which bf16 makes 0.25.  Over values in
    [1, 2) the results' own rounding (2^-9 of them, at random) averages out over 4096 of them to 2e-5; a sum of the rounded weights would
    be 2.4e-3 off in all of them."""
    g = torch.Generator().manual_seed(15)
    c = build(g, [(256, 257)] * 4, 8, 8, 16)
    D, hq = 128, 8
    c["qkv"][:] = 0
    c["qkv"][:, : hq * D].view(4, hq, D)[..., :2] = 1.0
    c["v"][:] = (1.0 + torch.rand(c["v"].shape, generator=g)).to(torch.bfloat16)
    c["k"][:] = 0
    c["k"][..., 0], c["k"][..., 1] = -15.625, -0.03125
    for row in c["rows"]:
        c["k"][c["table"][row, 0].long()] = 0
    out = run(ops, dev, c, impl).double()
    w = math.exp(-15.65625 * D ** -0.5)
    assert float(torch.tensor(w).bfloat16()) == 0.25
    for b, row in enumerate(c["rows"]):
        v = c["v"][c["table"][row, :257].long()].double()
        ref = (v[0] + 0.25 * v[1:].sum(0)) / (1.0 + 256 * w)
        assert abs(float(((out[b] - ref) / ref).mean())) < 3e-4


@pytest.mark.parametrize("hq,hkv,specs,ranges,dtype", [
    (16, 8, [(2000, 2100)], None, torch.bfloat16),             # a short portion after a long one
    (5, 1, [(0, 2060)], None, torch.bfloat16),                 # the first tiles' jobs have one range
    (10, 2, [(1100, 1101), (0, 129), (2000, 2160)], None, torch.float16),  # ragged ends, jobs of every number of ranges
    (6, 3, [(0, 5), (960, 1024)], (2, 3), torch.bfloat16),     # the last range takes what is left
    (4, 4, [(4000, 4100)], (64, 1), torch.bfloat16),           # 65 tiles, the most ranges
    (4, 2, [(64, 192), (0, 65)], (2, 1), torch.bfloat16),      # a wave's rows see nothing of their second range
])
def test_prefill_key_ranges(ops, dev, monkeypatch, hq, hkv, specs, ranges, dtype):
    """Ranges of the keys on workgroups of their own: the oracle's results; a job of one range keeps the bits of the launch without."""
    c = build(torch.Generator().manual_seed(16), specs, hq, hkv, 16, dtype)
    whole = run(ops, dev, c)
    tiles = sum(-(-n // ops.prefill_q_tile()) for n in c["q_lens"])
    rule = ops.prefill_ranges(tiles, hq, max(c["q_lens"]), max(c["k_lens"]))
    ranges = ranges or rule
    assert ranges[0] > 1
    ws = torch.empty(ops.prefill_ranges_workspace_bytes(tiles * hq * ranges[0]), dtype=torch.uint8, device=dev)
    plain = ops.attn_prefill
    monkeypatch.setattr(ops, "attn_prefill", lambda *a, **k: plain(*a, **k, ranges=ranges, workspace=ws))
    out = run(ops, dev, c)
    torch.testing.assert_close(out.double(), oracle(c), **TOL)
    assert torch.equal(out, run(ops, dev, c, order=None))
    at = 0
    for n, k in zip(c["q_lens"], c["k_lens"]):
        for t in range(0, n, 128):
            rows = slice(at + t, at + min(t + 128, n))
            if -(-(k - n + min(t + 128, n)) // 64) <= ranges[1]:
                assert torch.equal(out[rows], whole[rows])
        at += n


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("more", [0, 5, 12])
def test_prefill_short_tiles(ops, dev, more, dtype):
    """q tiles around the numbers of rows from which they are loaded and stored in whole rows, waves without rows among them, in launches of 400, 600 and 880
    workgroups (one round; one and a half, where such waves stay; more): the bits of the register-staged kernel, which has one way only."""
    new = [1, 31, 32, 33, 63, 64, 65, 127, 128, 96] + [129] * (more // 2) + [70] * (more % 2)
    c = build(torch.Generator().manual_seed(23), [(70, 70 + n) for n in new], 40, 8, 16, dtype)
    assert torch.equal(run(ops, dev, c, impl=4), run(ops, dev, c, impl=2))


@pytest.mark.parametrize("hq,hkv,specs,dtype", [
    (2, 1, [(0, 1)], torch.bfloat16),                                          # one row, one pair
    (16, 8, [(0, n) for n in (5, 31, 33, 64, 127, 129, 300)], torch.bfloat16),  # one tile, odd and even chains, waves without rows
    (6, 1, [(0, 129), (700, 701), (63, 192)], torch.float16),                  # three pairs of a kv head, a short portion after a long one
    (64, 8, [(1000, 1600)], torch.bfloat16),                                   # several pairs of a kv head, keys before the portion
    # more workgroups than compute units, whose lists go in turns: one XCD's kv heads shared by four, by two XCDs and one of its own several of them
    (16, 2, [(0, 900), (100, 1500), (0, 130), (0, 1000), (50, 650), (0, 300)], torch.bfloat16),
    (24, 6, [(0, 700), (300, 1100), (0, 129), (64, 650), (0, 1), (500, 1300)], torch.float16),
    (64, 16, [(0, 1), (700, 1000), (0, 520)], torch.float16),
])
def test_prefill_heads_in_pairs(ops, dev, monkeypatch, hq, hkv, specs, dtype):
    """Two heads a workgroup: the bits of one head a workgroup, which the oracle's tests pin; an odd group is refused."""
    c = build(torch.Generator().manual_seed(17), specs, hq, hkv, 16, dtype)
    whole = run(ops, dev, c)
    plain = ops.attn_prefill
    monkeypatch.setattr(ops, "attn_prefill", lambda *a, **k: plain(*a, **k, pairs=True))
    for order in ("heavy", "reversed", None):
        assert torch.equal(run(ops, dev, c, order=order), whole)
    with pytest.raises(RuntimeError, match="pairs"):
        run(ops, dev, build(torch.Generator().manual_seed(18), [(0, 5)], 5, 1, 16, dtype))


def test_prompt_attention_leaves_the_decode_workspace_alone(ops, dev):
    """Prompts and decode steps of one backend on different streams share no scratch: the sums of key ranges live in memory of their own."""
    from mini_sglang_amd.attention import HipAttnBackend
    from mini_sglang_amd.core import Batch, Context, Req
    from mini_sglang_amd.kvcache import create_kvcache_pool
    from mini_sglang_amd.model import ModelConfig

    old, new, hq, hkv = 2000, 100, 16, 8
    ctx = Context(16)
    m = ModelConfig(num_layers=1, num_qo_heads=hq, num_kv_heads=hkv, head_dim=128, hidden_size=1024, vocab_size=64, intermediate_size=64)
    ctx.page_table = torch.arange(2 * 2112, dtype=torch.int32, device=dev).view(2, 2112) % 2112
    ctx.kv_cache = create_kvcache_pool(m, 132, 16, torch.bfloat16, dev)
    for t in (ctx.kv_cache.k_tokens(0), ctx.kv_cache.v_tokens(0)):
        t.normal_()
    backend = HipAttnBackend(m, ctx)
    batch = Batch(reqs=[Req(input_ids=torch.zeros(old + new, dtype=torch.int32), table_idx=0, cached_len=old, output_len=1, uid=0)], phase="prefill")
    batch.out_loc = torch.arange(old, old + new, dtype=torch.int32, device=dev)
    batch.padded_reqs = batch.reqs
    backend.prepare_metadata(batch)
    assert batch.attn_metadata.ranges[0] > 1
    backend._workspace.fill_(0x5A)
    q, k, v = (torch.randn(new, h * 128, device=dev).bfloat16() for h in (hq, hkv, hkv))
    out = backend.forward(q.view(new, hq, 128), k, v, 0, batch)
    assert torch.isfinite(out).all() and bool((backend._workspace == 0x5A).all())


@pytest.mark.parametrize("hq,hkv,new,pairs", [(64, 8, 2048, True), (64, 8, 1900, True), (64, 8, 1700, False), (40, 8, 3072, False), (64, 8, 6144, True), (64, 8, 3328, False)])
def test_backend_pairs_heads_by_its_rule(ops, dev, monkeypatch, hq, hkv, new, pairs):
    """Heads go in pairs where a launch has 896 to 1024 chains of 15 tiles and more on average, or from 3072 of 36 on, and a kv head an even number of heads: the
    launch that the library gets is that one, and the bits are the other one's."""
    from mini_sglang_amd.attention import HipAttnBackend
    from mini_sglang_amd.core import Batch, Context, Req
    from mini_sglang_amd.kvcache import create_kvcache_pool
    from mini_sglang_amd.model import ModelConfig

    ctx = Context(16)
    width = max(3328, new)
    m = ModelConfig(num_layers=1, num_qo_heads=hq, num_kv_heads=hkv, head_dim=128, hidden_size=1024, vocab_size=64, intermediate_size=64)
    ctx.page_table = torch.arange(width, dtype=torch.int32, device=dev).view(1, width)
    ctx.kv_cache = create_kvcache_pool(m, width // 16, 16, torch.bfloat16, dev)
    backend = HipAttnBackend(m, ctx)
    batch = Batch(reqs=[Req(input_ids=torch.zeros(new, dtype=torch.int32), table_idx=0, cached_len=0, output_len=1, uid=0)], phase="prefill")
    batch.out_loc = torch.arange(new, dtype=torch.int32, device=dev)
    batch.padded_reqs = batch.reqs
    backend.prepare_metadata(batch)
    md = batch.attn_metadata
    assert md.pairs == pairs and md.ranges[0] == 1
    real, impls = ops.lib(), []

    class Recorder:
        def __getattr__(self, name):
            call = getattr(real, name)
            return call if name != "msgl_attn_prefill" else lambda *a: (impls.append(int(a[-2])), call(*a))[1]

    monkeypatch.setattr(ops, "lib", lambda: Recorder())
    q, k, v = (torch.randn(new, h * 128, device=dev).bfloat16() for h in (hq, hkv, hkv))
    out = backend.forward(q.view(new, hq, 128), k, v, 0, batch)
    md.pairs = not pairs and hq // hkv % 2 == 0  # the other launch, where there is one
    assert torch.equal(out, backend.forward(q.view(new, hq, 128), k, v, 0, batch))
    assert impls == [6 if pairs else 0, 6 if md.pairs else 0]


def test_a_small_decode_capacity_holds_the_small_batch_kernel(ops, dev):
    """The decode workspace is at least what small batches take, whatever number of pieces the caller asks for."""
    from mini_sglang_amd.attention import HipAttnBackend
    from mini_sglang_amd.core import Context
    from mini_sglang_amd.kvcache import create_kvcache_pool
    from mini_sglang_amd.model import ModelConfig

    for hq, hkv in ((16, 8), (8, 1), (64, 8)):
        ctx = Context(16)
        m = ModelConfig(num_layers=1, num_qo_heads=hq, num_kv_heads=hkv, head_dim=128, hidden_size=1024, vocab_size=64, intermediate_size=64)
        ctx.page_table = torch.zeros((70, 40960), dtype=torch.int32, device=dev)
        ctx.kv_cache = create_kvcache_pool(m, 4, 16, torch.bfloat16, dev)
        backend = HipAttnBackend(m, ctx, decode_capacity=70)
        for b in range(1, backend._small_heads // hkv + 1):
            need = ops.lib().msgl_attn_decode_small_workspace_bytes(b, ops.attn_decode_small_ranges(b, hkv, 40960), hq)
            assert backend._workspace.numel() >= need, (hq, hkv, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("hq,hkv", [(5, 1), (16, 8), (6, 3), (40, 8)])
@pytest.mark.parametrize("lens", [[1, 63, 64, 65, 127, 128, 129, 192, 2], [700], [257, 1000, 3] * 3, [1536]], ids=str)
def test_fresh_prompts_store_and_attend_in_one_launch(dev, dtype, hq, hkv, lens):
    """Requests with nothing cached: outputs and pool of the store and the attention one after the other, bit for bit; other slots stay; rows
    of two strides and key ranges take the two launches."""
    from mini_sglang_amd import attention, ops
    from mini_sglang_amd.core import Batch, Context, Req
    from mini_sglang_amd.kvcache import create_kvcache_pool
    from mini_sglang_amd.model import ModelConfig

    T, D, page = sum(lens), 128, 16
    g = torch.Generator(device=dev).manual_seed(T)
    pages = [-(-n // page) for n in lens]
    order = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(T)).to(dev)
    ctx = Context(page)
    ctx.page_table = torch.zeros((len(lens) + 1, (max(lens) + 31) // 32 * 32), dtype=torch.int32, device=dev)
    m = ModelConfig(1, hq, hkv, D, hq * D, 1024, 1024)
    ctx.kv_cache = create_kvcache_pool(m, sum(pages) + 1, page, dtype, dev)
    at, slots = 0, []
    for i, (n, c) in enumerate(zip(lens, pages)):
        s = (order[at: at + c, None] * page + torch.arange(page, device=dev)).reshape(-1)[:n]
        ctx.page_table[i, :n] = s.int()
        slots.append(s)
        at += c
    backend = attention.HipAttnBackend(m, ctx)
    qkv = torch.randn((T, (hq + 2 * hkv) * D), generator=g, device=dev).to(dtype)
    q, k, v = qkv.split([hq * D, hkv * D, hkv * D], dim=1)
    calls, real = [], attention.ops.attn_prefill_fresh

    def run(fresh, k, v, cached=0):
        batch = Batch(reqs=[Req(input_ids=torch.zeros(n, dtype=torch.int32), table_idx=i, cached_len=cached, output_len=8, uid=i) for i, n in enumerate(lens)], phase="prefill")
        batch.out_loc = torch.cat([s[cached:] for s in slots]).int()
        backend.prepare_metadata(batch)
        md = batch.attn_metadata
        assert md.fresh is (cached == 0)
        md.ranges, md.pairs, md.fresh = (1, 0), False, md.fresh and fresh
        ctx.kv_cache.pool.fill_(3.0)
        return backend.forward(q.view(T, hq, D), k, v, 0, batch), ctx.kv_cache.pool.clone(), batch

    try:
        attention.ops.attn_prefill_fresh = lambda *a, **kw: calls.append(1) or real(*a, **kw)
        want, pool, batch = run(False, k, v)
        assert not calls
        got, pool2, _ = run(True, k, v)
        assert len(calls) == 1
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)) and torch.equal(pool.view(torch.int16), pool2.view(torch.int16))
        got, pool2, _ = run(True, k, v.contiguous())  # rows of two strides
        assert len(calls) == 1 and torch.equal(got, want) and torch.equal(pool, pool2)
        batch.attn_metadata.ranges, batch.attn_metadata.fresh = (2, 1), True
        backend.forward(q.view(T, hq, D), k, v, 0, batch)
        assert len(calls) == 1
    finally:
        attention.ops.attn_prefill_fresh = real

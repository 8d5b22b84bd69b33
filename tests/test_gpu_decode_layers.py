"""msgl_decode_layers: a small decode batch's layers in one launch, against the same layers in float64 with and without the 16-bit rounding points."""
import math
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 1e-6


@pytest.fixture(scope="module")
def ops(dev):
    from mini_sglang_amd import ops as o

    return o


def _layer(g, dev, dtype, H, hq, hkv, inter, norm, ilv, ops):
    r = lambda *s, std=1.0, mean=0.0: (torch.randn(s, generator=g, device=dev) * std + mean).to(dtype)  # noqa: E731
    gate_up = r(2 * inter, H, std=H ** -0.5)
    w = SimpleNamespace(input_norm=r(H, std=0.1, mean=1.0), qkv=r((hq + 2 * hkv) * 128, H, std=H ** -0.5), q_norm=r(128, std=0.1, mean=1.0) if norm else None,
                        k_norm=r(128, std=0.1, mean=1.0) if norm else None, o=r(H, hq * 128, std=(hq * 128) ** -0.5), post_norm=r(H, std=0.1, mean=1.0),
                        gate_up=gate_up.index_select(0, ops.gate_up_interleave_index(inter, dev)) if ilv else gate_up, down=r(H, inter, std=inter ** -0.5))
    return w, gate_up


def _reference(x, layers, gate_ups, k_old, v_old, pos, cs, hq, hkv, rnd):
    """The layers in float64; rnd: the 16-bit rounding at the launches' rounding points, or nothing.  Returns y, residual, new keys and values per layer."""
    d = lambda t: t.double()  # noqa: E731
    G, B = hq // hkv, x.shape[0]
    cos, sin = d(cs[pos.long(), :64])[:, None, :], d(cs[pos.long(), 64:])[:, None, :]

    def norm(v, w):
        return rnd(v / torch.sqrt((v * v).mean(-1, keepdim=True) + EPS) * d(w))

    def rot(t):
        a, b = t[..., :64], t[..., 64:]
        return rnd(torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1))

    res, y, news = d(x), None, []
    for w, gu, ko, vo in zip(layers, gate_ups, k_old, v_old):
        v = res if y is None else res + y
        h, res = norm(v, w.input_norm), v if y is None else rnd(v)
        q, k, vv = rnd(h @ d(w.qkv).T).split([hq * 128, hkv * 128, hkv * 128], dim=1)
        q, k, vv = q.view(B, hq, 128), k.view(B, hkv, 128), vv.view(B, hkv, 128)
        if w.q_norm is not None:
            q, k = norm(q, w.q_norm), norm(k, w.k_norm)
        q, k = rot(q), rot(k)
        news.append((k, vv))
        out = []
        for b in range(B):
            kk, vb = torch.cat([d(ko[b]), k[b: b + 1]]), torch.cat([d(vo[b]), vv[b: b + 1]])
            sc = torch.einsum("hgd,nhd->hgn", q[b].view(hkv, G, 128), kk) * 128 ** -0.5
            out.append(torch.einsum("hgn,nhd->hgd", torch.softmax(sc, -1), vb).reshape(-1))
        v = rnd(rnd(torch.stack(out)) @ d(w.o).T) + res
        h, res = norm(v, w.post_norm), rnd(v)
        a = rnd(h @ d(gu).T)
        gate, up = a.chunk(2, dim=1)
        y = rnd(rnd(gate * torch.sigmoid(gate) * up) @ d(w.down).T)
    return y, res, news


def _case(ops, dev, dtype, H, hq, hkv, inter, lens, layers=3, page=16, norm=True, ilv=True, seed=0, ws=None):
    from mini_sglang_amd import flashinfer_compat as fi

    g = torch.Generator(device=dev).manual_seed(seed)
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
    loc = torch.stack([s[-1] for s in slots]).int()
    used = torch.zeros(pool, dtype=torch.bool, device=dev)
    for s in slots:
        used[s[:-1]] = True
    caches = []
    for _ in range(2 * layers):  # what lies in the new slots and in slots of no request must not be read into a result
        c = torch.randn((pool, hkv, 128), generator=g, device=dev).to(dtype)
        c[~used] = math.nan
        caches.append(c)
    kcs, vcs = caches[:layers], caches[layers:]
    made = [_layer(g, dev, dtype, H, hq, hkv, inter, norm, ilv, ops) for _ in range(layers)]
    x = torch.randn((B, H), generator=g, device=dev).to(dtype)
    seq = torch.tensor(lens, dtype=torch.int32, device=dev)
    cs = fi.build_cos_sin_cache(128, max(lens) + 1, 1e4, None, device=dev)
    before = [c.clone() for c in caches]
    args = (x, [w for w, _ in made], kcs, vcs, seq - 1, cs, loc, table, rows, seq)
    if ws is None:
        ws = torch.zeros(ops.decode_layers_workspace_bytes(B, layers, H, hq, hkv, inter), dtype=torch.uint8, device=dev)

    def launch(**kw):
        return ops.decode_layers(*args, ws, hq, ilv, EPS, 128 ** -0.5, **kw)

    y, res = launch()
    torch.cuda.synchronize()
    old = [[[c[s[:-1]] for s in slots] for c in before[i * layers: (i + 1) * layers]] for i in range(2)]
    ref = [_reference(x, [w for w, _ in made], [gu for _, gu in made], *old, seq - 1, cs, hq, hkv, f)
           for f in (lambda t: t, lambda t: t.to(dtype).double())]

    def far(a, b):
        return float((a.double() - b).norm() / b.norm())

    def check(got, i):
        """No further from the float64 layers than these with the rounding points, beyond what another order of sums moves (a quarter)."""
        got_e, ref_e = far(got, i(ref[0])), far(i(ref[1]), i(ref[0]))
        assert got_e <= 1.25 * ref_e + 1e-4 * torch.finfo(dtype).eps / 2 ** -8, (got_e, ref_e)

    check(y, lambda r: r[0])
    check(res, lambda r: r[1])
    rest = torch.ones(pool, dtype=torch.bool, device=dev)
    rest[loc.long()] = False
    for li in range(layers):
        for c, which in ((kcs[li], 0), (vcs[li], 1)):
            check(c[loc.long()], lambda r: r[2][li][which])
    for c, c0 in zip(caches, before):
        assert torch.equal(c[rest].view(torch.int16), c0[rest].view(torch.int16))
    stored = [c.clone() for c in caches]
    for _ in range(3):  # again over the rows that it stored
        y2, res2 = launch()
        assert torch.equal(y, y2) and torch.equal(res, res2) and all(torch.equal(a[loc.long()], b[loc.long()]) for a, b in zip(caches, stored))
    launch.ws, launch.before, launch.stored, launch.caches, launch.loc = ws, before, stored, caches, loc.long()
    return launch, y, res


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("lens", [[1], [533], [2100], [17, 16, 15], [700, 1, 40, 300, 5, 129, 2000, 64]], ids=str)
def test_layers_of_the_small_model(ops, dev, dtype, lens):
    _case(ops, dev, dtype, 1024, 16, 8, 3072, lens)


@pytest.mark.parametrize("H,hq,hkv,inter", [(256, 2, 1, 256), (256, 2, 2, 512), (512, 8, 1, 768), (1024, 6, 2, 2560), (768, 6, 3, 1280), (1024, 24, 4, 768)])
def test_layer_sizes(ops, dev, H, hq, hkv, inter):
    """Fewer groups of rows than workgroups, several tiles of rows a workgroup, one to eight query heads a kv head; without head norms, plain row order."""
    for lens, norm, ilv in (([90, 700], True, True), ([33], False, False)):
        assert ops.decode_layers_supported(len(lens), H, hq, hkv, inter)
        _case(ops, dev, torch.bfloat16, H, hq, hkv, inter, lens, layers=2, norm=norm, ilv=ilv)


def test_more_layers_than_a_launch_takes(ops, dev):
    _case(ops, dev, torch.bfloat16, 256, 2, 1, 256, [20, 9], layers=43)


def test_batches_share_a_workspace(ops, dev):
    ws = torch.zeros(ops.decode_layers_workspace_bytes(8, 3, 1024, 16, 8, 3072), dtype=torch.uint8, device=dev)
    for seed, lens in enumerate(([40], [300] * 8, [1200, 7], [90] * 5)):
        _case(ops, dev, torch.bfloat16, 1024, 16, 8, 3072, lens, seed=seed, ws=ws)


@pytest.mark.parametrize("H,hq,hkv,inter,lens", [(1024, 16, 8, 3072, [700, 90]), (1024, 16, 8, 3072, [300] * 7), (1024, 24, 4, 768, [40])])
def test_beside_other_work_on_the_device(ops, dev, H, hq, hkv, inter, lens):
    """Workgroups that find their CU taken are not waited for: the others do their share, with the same bits (of teams of a given size:
    test_small_teams)."""
    launch, y, res = _case(ops, dev, torch.bfloat16, H, hq, hkv, inter, lens)
    a = torch.randn((8192, 8192), device=dev, dtype=torch.bfloat16)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    for _ in range(10):
        with torch.cuda.stream(side):
            for _ in range(3):
                a @ a
        y2, res2 = launch()
        torch.cuda.synchronize()
        assert torch.equal(y, y2) and torch.equal(res, res2)


@pytest.mark.parametrize("H,hq,hkv,inter,lens", [(1024, 16, 8, 3072, [700, 90]), (1024, 16, 8, 3072, [2100, 300, 5, 17, 64, 129, 1, 40]), (1024, 24, 4, 768, [40]),
                                                 (512, 8, 1, 768, [1300, 3])])
def test_small_teams(ops, dev, H, hq, hkv, inter, lens):
    """Teams down to one workgroup: shares in several turns, weights fetched behind the rows, several (request, kv head, range) tasks each; the full team's bits."""
    launch, y, res = _case(ops, dev, torch.bfloat16, H, hq, hkv, inter, lens)
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    for most in (1, 2, 3, 31, 64, 130, cus - 1, cus):
        for c, c0 in zip(launch.caches, launch.before):
            c.copy_(c0)
        y2, res2 = launch(most=most)
        torch.cuda.synchronize()
        first, *_, last = _team_sizes(launch.ws)
        assert last == most if most < cus - 1 else 130 < first <= last <= most
        assert torch.equal(y, y2) and torch.equal(res, res2) and all(torch.equal(a[launch.loc], b[launch.loc]) for a, b in zip(launch.caches, launch.stored)), most


def _team_sizes(ws, layers=3):
    """What the last launch's first workgroup told the others, by layer: from the word that says that the team stays as it is on, that size."""
    sizes = []
    for word, _ in ws[256: 256 + 8 * layers].view(torch.int32).view(-1, 2).tolist():
        sizes.append(word >> 1)
        if word & 1:
            return sizes + [word >> 1] * (layers - len(sizes))
    raise AssertionError("a team that never stays")


@pytest.mark.parametrize("H,hq,hkv,inter,lens", [(1024, 16, 8, 3072, [700, 90]), (1024, 16, 8, 3072, [2100, 300, 5, 17, 64, 129, 1, 40]), (1024, 24, 4, 768, [40]),
                                                 (256, 2, 2, 512, [1300, 3, 5])])
def test_latecomers_join(ops, dev, H, hq, hkv, inter, lens):
    """Workgroups that come late take part from a later layer on (here: from the second or the third of three), with the bits of a team that was there at once."""
    launch, y, res = _case(ops, dev, torch.bfloat16, H, hq, hkv, inter, lens)
    for most, until in ((1, 1), (1, 2), (3, 1), (64, 2), (130, 1), (200, 2)):
        for c, c0 in zip(launch.caches, launch.before):
            c.copy_(c0)
        y2, res2 = launch(most=most, until=until)
        torch.cuda.synchronize()
        sizes = _team_sizes(launch.ws)
        assert sizes[:until] == [most] * until and sizes[-1] > 200, sizes
        assert torch.equal(y, y2) and torch.equal(res, res2) and all(torch.equal(a[launch.loc], b[launch.loc]) for a, b in zip(launch.caches, launch.stored)), most
    assert not ops.decode_layers_failed(launch.ws).any()


def test_launch_numbers_start_again(ops, dev):
    """The last number's launch clears packets and teams' sizes: none of an earlier launch could pass for one of a later launch with the same number."""
    launch, y, res = _case(ops, dev, torch.bfloat16, 1024, 16, 8, 3072, [700, 90])
    number, packets = launch.ws[128:132].view(torch.int32), launch.ws[256:].view(torch.int64)
    number.fill_(-3)
    for want in (-2, -1, 1, 2):
        y2, res2 = launch()
        assert int(number[0]) == want and torch.equal(y, y2) and torch.equal(res, res2)
        assert bool(packets.any()) == (want != -1)


@pytest.mark.parametrize("H,hq,hkv,inter,lens", [(1024, 16, 8, 3072, [700, 90]), (1024, 16, 8, 3072, [300] * 7), (512, 8, 1, 768, [40, 3])])
def test_waits_that_end_are_not_silent(ops, dev, H, hq, hkv, inter, lens):
    """A workgroup leaves without a word and the others give up waiting for it: every row has NaN, no wrong key or value is stored, the error word stays; the
    next launch is a launch like any other."""
    launch, y, res = _case(ops, dev, torch.bfloat16, H, hq, hkv, inter, lens)
    assert not ops.decode_layers_failed(launch.ws).any()
    for absent in (0, 1, 17):
        for c, c0 in zip(launch.caches, launch.before):
            c.copy_(c0)
        bad = sum(launch(looks=256, absent=absent))
        assert bad.isnan().any(dim=1).all()
        for c, c0, c1 in zip(launch.caches, launch.before, launch.stored):
            rows, old, new = (t[launch.loc] for t in (c, c0, c1))
            assert (rows.isnan() | (rows.view(torch.int16) == old.view(torch.int16)) | (rows == new)).all()
        for _ in range(2):
            y2, res2 = launch()
            assert torch.equal(y, y2) and torch.equal(res, res2) and all(torch.equal(a[launch.loc], b[launch.loc]) for a, b in zip(launch.caches, launch.stored))
        assert ops.decode_layers_failed(launch.ws).all()


@pytest.mark.parametrize("batch", [1, 3, 8])
def test_captured_steps_of_an_engine(dev, batch):
    """An engine whose steps take the launch: every replay gives the eager step's bits."""
    from mini_sglang_amd import attention, ops as o
    from mini_sglang_amd.core import Batch, Req
    from mini_sglang_amd.engine import Engine, EngineConfig
    from mini_sglang_amd.model import ModelConfig

    m = ModelConfig(3, 16, 8, 128, 1024, 4096, 3072, tie_word_embeddings=True, max_position=4096)
    eng = Engine(EngineConfig(model=m, max_running_req=batch, cuda_graph_bs=[batch], page_size=16, num_page_override=batch * 64, max_seq_len_override=1000), dev)
    eng.kv_cache.pool.normal_()
    eng.page_table[:batch] = torch.randperm(batch * 1024, device=dev)[: batch * eng.page_table.shape[1]].view(batch, -1).int()
    calls, real = [], attention.HipAttnBackend.decode_layers
    try:
        attention.HipAttnBackend.decode_layers = lambda self, *a: calls.append(1) or real(self, *a)
        for i in range(4):
            lens = [17 + 29 * i + 100 * b for b in range(batch)]
            reqs = [Req(input_ids=torch.zeros(n, dtype=torch.int32), table_idx=b, cached_len=n - 1, output_len=8, uid=b) for b, n in enumerate(lens)]
            step = Batch(reqs=reqs, phase="decode")
            eng.graph_runner.pad_batch(step)
            step.input_ids = torch.arange(7 * i, 7 * i + batch, dtype=torch.int32, device=dev)
            step.positions = torch.tensor(lens, dtype=torch.int32, device=dev) - 1
            step.out_loc = torch.stack([eng.page_table[b, n - 1] for b, n in enumerate(lens)])
            eng.attn_backend.prepare_metadata(step)
            got = eng.forward_logits(step).clone()
            for r, n in zip(reqs, lens):
                r.cached_len = n - 1
            with eng.ctx.forward_batch(step):
                want = eng.model.forward(eng.ctx, step)
            assert torch.equal(got, want)
        assert len(calls) == 4  # (the eager ones; the captured one was made by the engine)
        assert o.decode_layers_supported(batch, 1024, 16, 8, 3072)
        for _ in range(130):  # the error word reaches the host
            eng.attn_backend.prepare_metadata(step)
            torch.cuda.synchronize()
        o.decode_layers_failed(next(iter(eng.attn_backend._layers_workspaces.values()))).fill_(7)
        with pytest.raises(Exception, match="gave up"):
            for _ in range(130):
                eng.attn_backend.prepare_metadata(step)
                torch.cuda.synchronize()
    finally:
        attention.HipAttnBackend.decode_layers = real
        eng.shutdown()


def test_refusals(ops, dev):
    assert not ops.decode_layers_supported(9, 1024, 16, 8, 3072) and not ops.decode_layers_supported(1, 1000, 16, 8, 3072)
    assert not ops.decode_layers_supported(1, 5120, 40, 8, 17408) and not ops.decode_layers_supported(1, 2048, 16, 8, 2048)
    with pytest.raises(Exception):
        ops.decode_layers_workspace_bytes(0, 1, 1024, 16, 8, 3072)

"""GPU parity: greedy argmax (bit exact), temperature softmax, top-k / top-p sampling.

The reference's RNG stream (flashinfer) cannot be reproduced, so non-greedy sampling is checked
distributionally (chi-square against the exact filtered distribution of the oracle) plus exactness
on degenerate rows (top_k = 1, top_p -> 0  =>  argmax), as SURVEY.md Appendix B prescribes.
"""
import math

import pytest
import torch

from oracle import ref_ops

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops(dev):
    from mini_sglang_amd import ops as _ops

    return _ops


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("rows,vocab", [(1, 151936), (256, 151936), (7, 128256), (3, 1000), (5, 8), (2, 33333)])
def test_argmax_first_max_index(ops, dev, dtype, rows, vocab):
    g = torch.Generator().manual_seed(rows + vocab)
    logits = torch.randn((rows, vocab), generator=g).to(dtype)
    # force ties: duplicate the max at a later index -> the first one must win
    for r in range(rows):
        i = int(torch.argmax(logits[r].float()))
        if i + 1 < vocab:
            logits[r, vocab - 1] = logits[r, i]
    out = ops.argmax_rows(logits.to(dev))
    assert torch.equal(out.cpu(), ref_ops.argmax_ref(logits))


def test_argmax_strided_rows(ops, dev):
    """The graph path samples from logits[:B] of a wider fp32 buffer (P/engine/graph.py:33,165)."""
    g = torch.Generator().manual_seed(0)
    buf = torch.randn((8, 1000 + 24), generator=g)
    view = buf[:, :1000]
    out = ops.argmax_rows(view.to(dev)[:, :1000])
    assert torch.equal(out.cpu(), ref_ops.argmax_ref(view))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_softmax_temperature(ops, dev, dtype):
    g = torch.Generator().manual_seed(1)
    logits = (torch.randn((16, 151936), generator=g) * 3).to(dtype)
    t = torch.tensor([1e-6, 0.1, 0.6, 1.0, 2.0, 0.3, 0.9, 1.5] * 2, dtype=torch.float32)
    probs = ops.softmax_temperature(logits.to(dev), t.to(dev)).cpu()
    ref = ref_ops.softmax_temperature_ref(logits, t)
    torch.testing.assert_close(probs.double(), ref, atol=1e-6, rtol=2e-4)
    torch.testing.assert_close(probs.sum(-1), torch.ones(16), atol=1e-4, rtol=0)


def test_sampling_degenerate_rows_are_argmax(ops, dev):
    g = torch.Generator().manual_seed(2)
    V = 151936
    probs = torch.softmax(torch.randn((6, V), generator=g) * 2, -1)
    pd = probs.to(dev)
    am = ref_ops.argmax_ref(probs)
    k1 = torch.ones(6, dtype=torch.int32, device=dev)
    assert torch.equal(ops.sample_top_k_top_p(pd, k1, None, 42, 0).cpu(), am)
    p0 = torch.full((6,), 1e-6, dtype=torch.float32, device=dev)
    assert torch.equal(ops.sample_top_k_top_p(pd, None, p0, 42, 0).cpu(), am)
    assert torch.equal(ops.sample_top_k_top_p(pd, k1, p0, 7, 123).cpu(), am)


def test_sampling_is_deterministic_in_seed_and_offset(ops, dev):
    g = torch.Generator().manual_seed(3)
    probs = torch.softmax(torch.randn((64, 32000), generator=g), -1).to(dev)
    a = ops.sample_top_k_top_p(probs, None, None, 42, 100)
    b = ops.sample_top_k_top_p(probs, None, None, 42, 100)
    c = ops.sample_top_k_top_p(probs, None, None, 42, 164)
    assert torch.equal(a, b) and not torch.equal(a, c)


def _chi2_ok(counts, expected_p, n):
    keep = expected_p > 0
    assert counts[~keep].sum() == 0, "sampled a token outside the filtered support"
    # merge tiny cells
    e = expected_p[keep] * n
    o = counts[keep].double()
    order = torch.argsort(e, descending=True)
    e, o = e[order], o[order]
    big = e >= 5
    e2 = torch.cat([e[big], e[~big].sum().view(1)])
    o2 = torch.cat([o[big], o[~big].sum().view(1)])
    ok = e2 > 0
    chi2 = (((o2 - e2) ** 2)[ok] / e2[ok]).sum().item()
    dof = int(ok.sum()) - 1
    # mean dof, variance 2 dof; 6 sigma bound keeps the test stable yet sharp
    assert chi2 < dof + 6 * (2 * max(dof, 1)) ** 0.5 + 10, (chi2, dof)


@pytest.mark.parametrize("top_k,top_p", [(None, None), (50, None), (None, 0.9), (20, 0.7), (5, 0.99)])
def test_sampling_distribution(ops, dev, top_k, top_p):
    """Draw N samples of ONE row (replicated), compare frequencies with the oracle's filtered
    distribution."""
    g = torch.Generator().manual_seed(5)
    V, N = 4096, 40000
    row = torch.softmax(torch.randn(V, generator=g) * 2.5, -1)
    probs = row.unsqueeze(0).repeat(N, 1).to(dev)
    tk = None if top_k is None else torch.full((N,), top_k, dtype=torch.int32, device=dev)
    tp = None if top_p is None else torch.full((N,), top_p, dtype=torch.float32, device=dev)
    out = ops.sample_top_k_top_p(probs, tk, tp, 1234, 0).cpu().long()
    assert out.min() >= 0 and out.max() < V
    counts = torch.bincount(out, minlength=V)
    expect = ref_ops.top_k_top_p_filter_ref(row.unsqueeze(0), None if top_k is None else [top_k],
                                            None if top_p is None else [top_p])[0]
    _chi2_ok(counts, expect, N)


def test_sampling_per_row_parameters(ops, dev):
    """Different (k, p) per row, as Sampler.prepare builds them (P/engine/sample.py:53-68)."""
    g = torch.Generator().manual_seed(6)
    V = 151936
    probs = torch.softmax(torch.randn((8, V), generator=g) * 3, -1)
    ks = [1, 5, V, 50, 1000, V, 2, 10]
    ps = [1.0, 0.5, 0.3, 1.0, 0.9, 1e-6, 0.99, 0.1]
    support = ref_ops.top_k_top_p_filter_ref(probs, ks, ps) > 0
    pd = probs.to(dev)
    tk = torch.tensor(ks, dtype=torch.int32, device=dev)
    tp = torch.tensor(ps, dtype=torch.float32, device=dev)
    for off in range(0, 80, 8):
        out = ops.sample_top_k_top_p(pd, tk, tp, 99, off).cpu().long()
        for r in range(8):
            assert support[r, out[r]], (r, int(out[r]))


# ---------------------------------------------------------------- fused softmax + draw (temperature only)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("temperature", [0.6, 1.0, 1.7])
def test_sample_from_logits_distribution(ops, dev, dtype, temperature):
    """One row replicated N times: frequencies of the fused kernel against softmax(logits / T) of the oracle."""
    g = torch.Generator().manual_seed(11)
    V, N = 4096, 40000
    logits = (torch.randn(V, generator=g) * 2.5).to(dtype)
    t = torch.full((N,), temperature, dtype=torch.float32)
    out = ops.sample_from_logits(logits.unsqueeze(0).repeat(N, 1).to(dev), t.to(dev), 4321, 0).cpu().long()
    assert out.min() >= 0 and out.max() < V
    expect = ref_ops.softmax_temperature_ref(logits.unsqueeze(0), t[:1])[0]
    _chi2_ok(torch.bincount(out, minlength=V), expect, N)


@pytest.mark.parametrize("vocab", [151936, 128256, 33336, 1000, 8])
def test_sample_from_logits_edges(ops, dev, vocab):
    """T -> 0 rows return the (unique) argmax; results are a function of (seed, offset) only; the graph path's
    fp32 buffer view (row stride > vocab) and a ragged last wave segment are covered by the vocab list."""
    g = torch.Generator().manual_seed(vocab)
    rows = 6
    pad = 24 if vocab % 8 == 0 else 0
    buf = torch.randn((rows, vocab + pad), generator=g) * 3
    logits = buf[:, :vocab]
    dl = buf.to(dev)[:, :vocab]
    cold = torch.full((rows,), 1e-6, dtype=torch.float32, device=dev)
    assert torch.equal(ops.sample_from_logits(dl, cold, 42, 0).cpu(), ref_ops.argmax_ref(logits))
    warm = torch.full((rows,), 0.8, dtype=torch.float32, device=dev)
    a = ops.sample_from_logits(dl, warm, 42, 100)
    b = ops.sample_from_logits(dl, warm, 42, 100)
    assert torch.equal(a, b) and int(a.min()) >= 0 and int(a.max()) < vocab
    draws = torch.stack([ops.sample_from_logits(dl, warm, 42, 1000 + 8 * i) for i in range(12)])
    if vocab > 8:
        assert len(set(draws[:, 0].tolist())) > 1  # the offset moves the Philox stream


def test_sample_from_logits_matches_probs_path_statistically(ops, dev):
    """Same logits through softmax -> sampling_from_probs and through the fused kernel: the two empirical
    distributions agree (two-sample chi-square on the pooled top cells)."""
    g = torch.Generator().manual_seed(17)
    V, N = 2048, 30000
    logits = torch.randn(V, generator=g) * 2
    t = torch.full((N,), 0.6, dtype=torch.float32, device=dev)
    dl = logits.unsqueeze(0).repeat(N, 1).to(dev)
    a = torch.bincount(ops.sample_from_logits(dl, t, 5, 0).cpu().long(), minlength=V).double()
    b = torch.bincount(ops.sample_top_k_top_p(ops.softmax_temperature(dl, t), None, None, 6, 0).cpu().long(),
                       minlength=V).double()
    big = (a + b) >= 20
    chi2 = (((a - b) ** 2)[big] / (a + b)[big]).sum().item()
    dof = int(big.sum()) - 1
    assert chi2 < dof + 6 * (2 * dof) ** 0.5 + 10, (chi2, dof)


def test_top_k_larger_than_the_number_of_positive_probabilities(ops, dev):
    """ADVICE r1 (sampling.hip:249): a low-temperature softmax underflows the tail to exactly 0; with top_k above
    the count of positive entries the count search finds no bin and must behave as 'keep every positive entry'
    (what flashinfer returns), also when top_p follows.  The sample can only ever be a positive-probability index."""
    V = 151936
    g = torch.Generator().manual_seed(5)
    probs = torch.zeros((6, V), dtype=torch.float32)
    hot = [int(torch.randint(0, V, (1,), generator=g)) for _ in range(6)]
    for r, h in enumerate(hot):
        probs[r, h] = 1.0                      # rows 0-2: one positive entry (T = 1e-6 on a non-greedy row)
    for r in (3, 4, 5):                        # rows 3-5: three positive entries, k = 50
        probs[r] = 0
        probs[r, hot[r]] = 0.7
        probs[r, (hot[r] + 17) % V] = 0.2
        probs[r, (hot[r] + 40000) % V] = 0.1
    pd = probs.to(dev)
    k = torch.full((6,), 50, dtype=torch.int32, device=dev)
    p = torch.tensor([0.9, 1e-6, 1.0, 0.5, 0.95, 1.0], dtype=torch.float32, device=dev)
    allowed = [set(torch.nonzero(probs[r]).flatten().tolist()) for r in range(6)]
    seen = [set() for _ in range(6)]
    for it in range(40):
        for kk, pp in ((k, p), (k, None)):
            out = ops.sample_top_k_top_p(pd, kk, pp, seed=11, offset=it * 6).cpu().tolist()
            for r, o in enumerate(out):
                assert o in allowed[r], (r, o)
                if pp is None:
                    seen[r].add(o)
    for r in range(3):
        assert seen[r] == {hot[r]}
    # row 3 with top_p = 0.5 keeps only the 0.7 entry; without top_p all three positives are reachable
    outs = [ops.sample_top_k_top_p(pd, k, p, seed=3, offset=i * 6).cpu().tolist()[3] for i in range(30)]
    assert set(outs) == {hot[3]}
    assert len(seen[5]) >= 2


def _philox(seed, ctr):
    """First word of Philox4x32-10 of counter (ctr, 0) under key `seed`."""
    c, k = [ctr & 0xFFFFFFFF, ctr >> 32, 0, 0], [seed & 0xFFFFFFFF, seed >> 32]
    for _ in range(10):
        a, b = 0xD2511F53 * c[0], 0xCD9E8D57 * c[2]
        c = [(b >> 32) ^ c[1] ^ k[0], b & 0xFFFFFFFF, (a >> 32) ^ c[3] ^ k[1], a & 0xFFFFFFFF]
        k = [(k[0] + 0x9E3779B9) & 0xFFFFFFFF, (k[1] + 0xBB67AE85) & 0xFFFFFFFF]
    return c[0]


def _filtered_pick(p, k, pp, seed, ctr):
    """The pick over one row of fp32 probabilities in whole numbers of 2^-40: k-th largest value, then the value where the descending
    mass reaches pp of what is kept (ties stay), then the inverse CDF in index order."""
    import numpy as np

    mass = np.floor(np.where(p > 0, p, 0).astype(np.float64) * 2.0 ** 40).astype(np.int64)
    keep = p > 0
    if 1 <= k < p.size and keep.sum() >= k:
        keep &= p >= np.sort(p[keep])[-k]
    total = int(mass[keep].sum())
    if pp < 1.0 and total > 0:
        target = min(max(int(float(np.float32(pp)) * float(total)), 1), total)
        order = np.argsort(-p[keep], kind="stable")
        v = p[keep][order][int(np.searchsorted(np.cumsum(mass[keep][order]), target))]
        keep &= p >= v
        total = int(mass[keep].sum())
    u = (total * _philox(seed, ctr)) >> 32
    idx = np.nonzero(keep)[0]
    run = np.cumsum(mass[idx])
    return int(idx[np.searchsorted(run, u, side="right")]) if total else 0


# vocabularies around the 1024 columns and the strips of 8 loads; rows whose largest numbers share one column (the candidate list
# overflows or asks for more than its column maxima give), plain rows, ties, few positive probabilities
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("vocab", [1, 7, 1023, 1025, 8192 + 5, 33333, 151936])
def test_filtered_draw_is_the_integer_rule(ops, dev, dtype, vocab):
    g = torch.Generator().manual_seed(vocab)
    rows = [(k, p, t, kind) for kind in ("plain", "column", "ties", "cold")
            for k, p, t in ((1, 1.0, 1.0), (50, 0.9, 0.7), (0, 0.8, 0.5), (0, 0.99, 1.0), (1024, 0.95, 1.0), (1500, 0.9, 1.0), (20, 1.0, 0.4), (0, 1.0, 1.0))]
    logits = torch.randn((len(rows), vocab), generator=g) * 2.5
    for r, (_, _, _, kind) in enumerate(rows):
        if kind == "column":
            logits[r, 3::1024] += 9.0
        elif kind == "ties":
            logits[r] = torch.round(logits[r] * 2) / 2
        elif kind == "cold":
            logits[r, 5:] -= 300.0
    logits = logits.to(dtype).to(dev)
    k = torch.tensor([x[0] for x in rows], dtype=torch.int32, device=dev)
    p = torch.tensor([x[1] for x in rows], dtype=torch.float32, device=dev)
    t = torch.tensor([x[2] for x in rows], dtype=torch.float32, device=dev)
    probs = ops.softmax_temperature(logits, t)
    host = probs.cpu().numpy()
    for off in (0, 1000):
        want = [_filtered_pick(host[r], rows[r][0], rows[r][1], 77, off + r) for r in range(len(rows))]
        assert ops.sample_top_k_top_p(probs, k, p, 77, off).cpu().tolist() == want
        assert ops.sample_filtered_logits(logits, t, k, p, 77, off).cpu().tolist() == want


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
def test_a_second_draw_takes_what_the_first_one_took(ops, dev, dtype):
    """Several draws from one softmax() result while the logits and temperatures buffers go on to the next step: all from the first step's
    probabilities, and so is .probs()."""
    from mini_sglang_amd import flashinfer_compat as fi

    g = torch.Generator().manual_seed(9)
    step = [(torch.randn((5, 33333), generator=g) * 2.5).to(dtype).to(dev) for _ in range(2)]
    buf = torch.empty((5, 33400), dtype=dtype, device=dev)[:, :33333]  # rows with a stride, as of a padded buffer
    temp = [torch.full((5,), x, device=dev) for x in (0.7, 0.3)]
    k, p = torch.full((5,), 40, dtype=torch.int32, device=dev), torch.full((5,), 0.9, device=dev)
    t = temp[0].clone()
    buf.copy_(step[0])
    draw = type(fi.sampling)()
    probs = draw.softmax(buf, t)
    got = [draw.top_k_top_p_sampling_from_probs(probs, k, p)]
    buf.copy_(step[1])
    t.copy_(temp[1])
    got += [draw.top_k_sampling_from_probs(probs, k), draw.top_p_sampling_from_probs(probs, p)]
    stored = ops.softmax_temperature(step[0], temp[0])
    want = [ops.sample_top_k_top_p(stored, a, b, torch.initial_seed(), 5 * i) for i, (a, b) in enumerate(((k, p), (k, None), (None, p)))]
    assert torch.stack(got).tolist() == torch.stack(want).tolist()
    assert torch.equal(probs.probs(), stored)


@pytest.mark.parametrize("vocab", [2000, 33333])
def test_nucleus_at_the_list_s_length(ops, dev, vocab):
    """Nuclei of 1 to 130 tokens around the 64 that the candidate list is asked for, equal and unequal ones, in different columns and in one: the
    picks of the integer rule, from the logits and from stored probabilities."""
    g = torch.Generator().manual_seed(vocab)
    sizes = [1, 2, 60, 63, 64, 65, 66, 70, 100, 130]
    rows = [(m, kind) for m in sizes for kind in ("equal", "steps", "column")]
    logits = torch.full((len(rows), vocab), -9.0) + 0.1 * torch.randn((len(rows), vocab), generator=g)
    for r, (m, kind) in enumerate(rows):
        at = torch.randperm(vocab, generator=g)[:m] if kind != "column" else (torch.arange(m) * 1024 + 5) % vocab
        logits[r, at] = 8.0 if kind == "equal" else 8.0 - 0.03 * torch.arange(m)
    logits = logits.bfloat16().to(dev)
    t, p = torch.ones(len(rows), device=dev), torch.full((len(rows),), 0.98, device=dev)
    probs = ops.softmax_temperature(logits, t)
    host = probs.cpu().numpy()
    for off in (0, 5000, 10000):
        want = [_filtered_pick(host[r], 0, 0.98, 3, off + r) for r in range(len(rows))]
        assert ops.sample_filtered_logits(logits, t, None, p, 3, off).cpu().tolist() == want
        assert ops.sample_top_k_top_p(probs, None, p, 3, off).cpu().tolist() == want


# rows that 16, 8, 4, 2 and 1 workgroups share, with and without a top-k; vocabularies at the shortest rows that are shared, beside whole columns and
# chunks, and above 1024 chunks of 512; masses whose threshold lies high, in the tail, in a tie and (column) among numbers that the bound misses
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,vocab", [(3, 65536), (33, 33333), (40, 8192), (130, 8193), (257, 8200), (2, 600_003), (64, 98304), (17, 98309), (65, 98304),
                                        (130, 16391), (64, 16384), (9, 32000)])
def test_a_row_shared_by_workgroups_draws_the_same(ops, dev, dtype, rows, vocab):
    g = torch.Generator(device=dev).manual_seed(vocab)
    logits = torch.randn((rows, vocab), generator=g, device=dev) * 2.5
    for r in range(rows):
        if r % 5 == 1:
            logits[r, 3::1024] += 9.0
        elif r % 5 == 2:
            logits[r] = torch.round(logits[r] * 2) / 2
        elif r % 5 == 3:
            logits[r, 5:] -= 300.0
    logits = logits.to(dtype)
    t = torch.tensor([(0.5, 0.7, 1.0, 0.02)[r % 4] for r in range(rows)], device=dev)
    p = torch.tensor([(0.8, 0.98, 1e-6, 1.0, 0.999999, 0.5)[r % 6] for r in range(rows)], device=dev)
    k = torch.tensor([(40, 0, 1024, 1, 1500)[r % 5] for r in range(rows)], dtype=torch.int32, device=dev)
    probs = ops.softmax_temperature(logits, t)
    host = probs.cpu().numpy()
    for kk, pp in ((None, p), (k, p), (k, None), (None, None)):
        for off in (0, 1000):
            got = ops.sample_filtered_logits(logits, t, kk, pp, 77, off).cpu().tolist()
            assert got == ops.sample_top_k_top_p(probs, kk, pp, 77, off).cpu().tolist()
            if rows <= 33 and off == 0:
                ks, ps = ([0] * rows if kk is None else kk.tolist()), ([1.0] * rows if pp is None else pp.tolist())
                assert got == [_filtered_pick(host[r], ks[r], ps[r], 77, r) for r in range(rows)]
    if (vocab * logits.element_size()) % 16 == 0:  # the unfiltered draw from the logits: as its own rows one by one, each with more workgroups
        got = ops.sample_from_logits(logits, t, 5, 300).tolist()
        assert got == [int(ops.sample_from_logits(logits[r: r + 1], t[r: r + 1], 5, 300 + r)) for r in range(rows)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,vocab,gap", [(129, 32000, 0), (129, 32004, 4), (128, 32000, 0), (130, 40961, 7), (20, 163848, 0)])
def test_copies_of_shared_rows(ops, dev, dtype, rows, vocab, gap):
    """The rows and temperatures that a draw leaves for later ones are its inputs, bit for bit: above 128 rows from the kernel that sums them, else (and where
    16 bytes cannot be stored) beside the picks; rows of more tiles than are asked for ahead."""
    g = torch.Generator(device=dev).manual_seed(rows)
    logits = (torch.randn((rows, vocab + gap), generator=g, device=dev) * 2.5).to(dtype)[:, :vocab]
    t = torch.rand(rows, generator=g, device=dev) + 0.5
    p = torch.full((rows,), 0.9, device=dev)
    k = torch.full((rows,), 30, dtype=torch.int32, device=dev)
    for kk, pp in ((None, p), (k, p)):
        n = ops.lib().msgl_sample_workspace_bytes(rows, vocab, 1, kk is not None, 1)
        ws = torch.empty(max(n, 16), dtype=torch.uint8, device=dev)
        out = torch.empty(rows, dtype=torch.int32, device=dev)
        kept, kept_t = torch.full((rows * vocab + 64,), 7.0, dtype=dtype, device=dev), torch.zeros(rows, device=dev)
        ops.check(ops.lib().msgl_sample_filtered_logits_ws(
            out.data_ptr(), kept.data_ptr(), kept_t.data_ptr(), logits.data_ptr(), t.data_ptr(), None if kk is None else kk.data_ptr(), pp.data_ptr(), rows, vocab,
            logits.stride(0), ops._logits_dt(logits), 3, 0, ws.data_ptr() if n else None, n, ops._stream()), "sample")
        assert bool((kept[: rows * vocab].view(rows, vocab) == logits).all()) and bool((kept[rows * vocab:] == 7).all()) and bool((kept_t == t).all())
        assert out.tolist() == ops.sample_top_k_top_p(ops.softmax_temperature(logits, t), kk, pp, 3, 0).tolist()


def _draw_with_workspace(ops, dev, logits, t, k, p):
    """A shared-row draw with a workspace to look into: its first parts are 16 bytes a row (maximum, candidates' bound, ..) and 1024 maxima a row."""
    rows, vocab = logits.shape
    n = ops.lib().msgl_sample_workspace_bytes(rows, vocab, 1, k is not None, p is not None)
    assert n > 0
    ws, out = torch.zeros(n, dtype=torch.uint8, device=dev), torch.empty(rows, dtype=torch.int32, device=dev)
    ops.check(ops.lib().msgl_sample_filtered_logits_ws(
        out.data_ptr(), None, None, logits.data_ptr(), t.data_ptr(), None if k is None else k.data_ptr(), None if p is None else p.data_ptr(), rows, vocab,
        logits.stride(0), ops._logits_dt(logits), 1, 0, ws.data_ptr(), n, ops._stream()), "sample")
    torch.cuda.synchronize()
    at = (16 * rows + 255) // 256 * 256
    return ws[: 16 * rows].view(torch.int32).view(rows, 4), ws[at: at + 4096 * rows].view(torch.float32).view(rows, 1024)


@pytest.mark.parametrize("vocab", [100001, 98304, 131073])
def test_maxima_of_a_shared_row_are_of_different_numbers(ops, dev, vocab):
    """The k-th largest of the 1024 maxima bounds the k-th largest number from below only if no number counts twice; a row that the bound cuts short is
    drawn by radix levels, six times as slow.  All numbers differ, and a workgroup's last one is its largest."""
    rows = 4
    logits = torch.arange(vocab, device=dev, dtype=torch.float32).repeat(rows, 1).mul_(1e-3)
    t, k = torch.ones(rows, device=dev), torch.full((rows,), 20, dtype=torch.int32, device=dev)
    head, top = _draw_with_workspace(ops, dev, logits, t, k, None)
    for r in range(rows):
        real = top[r][top[r] > -math.inf]
        assert real.numel() == real.unique().numel() and real.numel() > 512


@pytest.mark.parametrize("temperature", [1.0, 0.25, 0.1])
def test_the_bound_of_candidates_reaches_low_temperatures(ops, dev, temperature):
    """The k-th largest weight of a sharp row (2^-29, 2^-115 and, at 0.1, none above 0) is bounded from below as long as there is one."""
    rows, vocab = 3, 131072
    logits = torch.full((rows, vocab), -4.0, device=dev)
    logits[:, ::1021] = 0.0
    logits[:, 777] = 20.0
    t, k = torch.full((rows,), temperature, device=dev), torch.full((rows,), 30, dtype=torch.int32, device=dev)
    head, _ = _draw_with_workspace(ops, dev, logits, t, k, None)
    weight = 2.0 ** (-20.0 / temperature * 1.4426950408889634)
    for bits in head[:, 1].tolist():
        if weight > 2.0 ** -126:
            bound = torch.tensor(bits, dtype=torch.int32).view(torch.float32).item()
            assert weight / 1.25 <= bound <= weight * 1.00001
        else:
            assert bits == 0


# (filter, rows, vocabulary) on both sides of the lines that split_of's comment gives times for
@pytest.mark.parametrize("how,rows,vocab,shared", [
    ("none", 64, 65536, True), ("none", 65, 65536, False), ("none", 128, 98303, False), ("none", 128, 98304, True), ("none", 129, 98304, False),
    ("k", 64, 98304, True), ("k", 1, 98303, False), ("k", 65, 151936, False),
    ("p", 1, 31999, False), ("p", 1, 32000, True), ("p", 63, 31999, False), ("p", 64, 16384, True), ("p", 64, 16383, False), ("p", 256, 16384, True), ("p", 257, 32000, False),
])
def test_draws_that_share_their_rows(ops, how, rows, vocab, shared):
    assert (ops.lib().msgl_sample_workspace_bytes(rows, vocab, how != "none", how == "k", how == "p") > 0) is shared


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,vocab", [(3, 65536), (64, 98304), (40, 151936), (1, 600_008), (70, 131080)])
def test_unfiltered_draws_of_shared_rows_are_those_of_one_workgroup(ops, dev, dtype, rows, vocab):
    """Rows that 16 to 2 workgroups share, more than 1024 chunks of 512 numbers among them, against the kernel with one workgroup a row (no workspace)."""
    g = torch.Generator(device=dev).manual_seed(rows + vocab)
    logits = (torch.randn((rows, vocab), generator=g, device=dev) * 2.5).to(dtype)
    t = torch.tensor([(0.5, 1.0, 3.0, 0.02)[r % 4] for r in range(rows)], device=dev)
    assert ops.lib().msgl_sample_workspace_bytes(rows, vocab, 0, 0, 0) > 0
    want = torch.empty(rows, dtype=torch.int32, device=dev)
    for off in range(0, 4000, 500):
        ops.check(ops.lib().msgl_sample_from_logits(want.data_ptr(), logits.data_ptr(), t.data_ptr(), rows, vocab, logits.stride(0), ops._logits_dt(logits), 9, off,
                                                    ops._stream()), "sample")
        assert torch.equal(ops.sample_from_logits(logits, t, 9, off), want)


# one launch for draws with a top-k: 4, 8 and 16 workgroups a row, unaligned rows, the largest share that fits the registers and one that does not
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,vocab", [(64, 98304), (64, 151936), (33, 163840), (33, 163848), (20, 98305), (5, 131071), (1, 151936)])
def test_draws_in_one_launch(ops, dev, dtype, rows, vocab):
    """The picks of stored probabilities, whether the workgroups wait for each other's maxima or (wait_us 0) look them up; copies bit for bit; the zeros that
    the next launch starts from are left."""
    g = torch.Generator(device=dev).manual_seed(rows + vocab)
    logits = torch.randn((rows, vocab), generator=g, device=dev) * 2.5
    for r in range(rows):
        if r % 5 == 1:
            logits[r, 3::1024] += 9.0  # the largest numbers in one column: more candidates than a list holds
        elif r % 5 == 2:
            logits[r] = torch.round(logits[r] * 2) / 2
        elif r % 5 == 3:
            logits[r, 5:] -= 300.0
    logits = logits.to(dtype)
    t = torch.tensor([(0.5, 0.7, 1.0, 0.02)[r % 4] for r in range(rows)], device=dev)
    p = torch.tensor([(0.8, 0.98, 1e-6, 1.0, 0.999999, 0.5)[r % 6] for r in range(rows)], device=dev)
    k = torch.tensor([(40, 0, 1024, 1, 1500, vocab)[r % 6] for r in range(rows)], dtype=torch.int32, device=dev)
    probs = ops.softmax_temperature(logits, t)
    kept = torch.empty_like(logits), torch.empty_like(t)
    for pp in (p, None):
        for off in (0, 1000):
            want = ops.sample_top_k_top_p(probs, k, pp, 77, off)
            for wait_us in (20, 0, 20):
                kept[0].zero_()
                got = ops.sample_filtered_logits(logits, t, k, pp, 77, off, keep=kept, wait_us=wait_us)
                assert torch.equal(got, want)
                assert torch.equal(kept[0].view(torch.uint8), logits.view(torch.uint8)) and torch.equal(kept[1], t)
    assert not any(bool(z.any()) for z in ops._SAMPLE_TEAMS.values())


def test_draws_in_one_launch_beside_others(ops, dev):
    """Workgroups without a place on the device are not waited for; streams do not share what the workgroups meet in; a captured draw has its own."""
    logits = (torch.randn((64, 151936), generator=torch.Generator(device=dev).manual_seed(1), device=dev) * 2.5).bfloat16()
    t, k, p = torch.ones(64, device=dev), torch.full((64,), 50, dtype=torch.int32, device=dev), torch.full((64,), 0.9, device=dev)
    want = ops.sample_top_k_top_p(ops.softmax_temperature(logits, t), k, p, 9, 0)
    graph = torch.cuda.CUDAGraph()
    ops.sample_filtered_logits(logits, t, k, p, 9, 0)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        captured = ops.sample_filtered_logits(logits, t, k, p, 9, 0)
    a = torch.randn((8192, 8192), device=dev, dtype=torch.bfloat16)
    sides = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    for i in range(10):
        captured.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(sides[0]):
            a @ a
            other = ops.sample_filtered_logits(logits, t, k, p, 9, 0)
        if i % 2:
            with torch.cuda.stream(sides[1]):
                graph.replay()
        else:
            graph.replay()
        got = ops.sample_filtered_logits(logits, t, k, p, 9, 0)
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(other, want) and torch.equal(captured, want)
    assert len(ops._SAMPLE_TEAMS) <= ops._SAMPLE_TEAMS_MAX

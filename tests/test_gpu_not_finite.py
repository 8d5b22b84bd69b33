"""What a number that is none reaches in the hybrid decoders' matrix-core kernels: the rows and columns that use it, nothing else."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
NEW, OLD = (300, 90, 1, 40), (40, 500, 77, 0)  # request 0 holds the number; its group of decoded or few tokens lies beside
LENS = [n + k for n, k in zip(NEW, OLD)]
AT = 205  # its position in request 0's sequence, inside a token group


@pytest.fixture
def dev():
    return torch.device("cuda:0")


def _latent(dev, key, value, q, table, rest):
    from mini_sglang_amd import mixops

    out = torch.empty((q.shape[0], 16, 512), device=dev)
    mixops.latent_attn(out, q[:, : 16 * 576].reshape(-1, 16, 576).contiguous(), key[:, :576].contiguous(), table, *rest, 512, 0.05, max_keys=max(LENS))
    return out.flatten(1)


def _window(dev, key, value, q, table, rest):
    from mini_sglang_amd import mixops

    out = torch.empty((q.shape[0], 16 * 128), dtype=torch.bfloat16, device=dev)
    talk = torch.eye(16, device=dev) + 0.1
    mixops.window_attn(out, q[:, : 16 * 129].bfloat16().contiguous(), 16 * 128, key[:, :512].contiguous(), value[:, :512].contiguous(), table, *rest, 16, 4, 128, 128, 0, 0.05, talk,
                       max_keys=max(LENS))
    return out


def _maps(dev, key, value, q, table, rest):
    from mini_sglang_amd import mixops

    out = torch.empty((q.shape[0], 16 * 128), dtype=torch.bfloat16, device=dev)
    mixops.diff_attn(out, q[:, : 16 * 128].contiguous(), key[:, :512].contiguous(), value[:, :512].contiguous(), table, *rest, 16, 4, 64, 128, 0.1, 0, 0,
                     torch.full((1,), 0.4, device=dev), 0.7, 1e-5, max_keys=max(LENS))
    return out


@pytest.mark.parametrize("call,group", [(_latent, 8), (_window, 16), (_maps, 32)], ids=["latent", "window", "maps"])
def test_attention_rows_that_a_number_reaches(dev, call, group):
    """A key with a NaN makes the rows that see it undefined and leaves all others their bits.  An infinite value does the same but for the rows of
    its own token group (zero times infinity in the product of weights and values)."""
    g = torch.Generator().manual_seed(11)
    slots, at = torch.randperm(sum(LENS), generator=g), 0
    table = torch.zeros((len(LENS), 600), dtype=torch.int32)
    for b, n in enumerate(LENS):
        table[b, :n] = slots[at: at + n].int()
        at += n
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)  # noqa: E731
    rest = i32(range(len(LENS))), i32(LENS), torch.tensor((0,) + NEW).cumsum(0).int().to(dev), len(LENS)
    key, value = (torch.randn(sum(LENS), 576, generator=g).bfloat16().to(dev) for _ in range(2))
    q = torch.randn(sum(NEW), 16 * 576, generator=g).to(dev)
    clean = call(dev, key, value, q, table.to(dev), rest)
    assert torch.isfinite(clean).all()
    row, slot = AT - OLD[0], int(table[0, AT])
    bad = key.clone()
    bad[slot, 550 if call is _latent else 5] = torch.nan  # (a latent row's first 512 columns are its value too)
    got = call(dev, bad, value, q, table.to(dev), rest)
    assert torch.equal(got[:row], clean[:row]) and torch.equal(got[NEW[0]:], clean[NEW[0]:])
    assert torch.isnan(got[row: NEW[0], 5]).all()
    bad = (key if call is _latent else value).clone()
    bad[slot, 5] = torch.inf
    got = call(dev, *((bad, value) if call is _latent else (key, bad)), q, table.to(dev), rest)
    before = row // group * group
    assert torch.equal(got[:before], clean[:before]) and torch.equal(got[NEW[0]:], clean[NEW[0]:])
    assert not torch.isfinite(got[row: NEW[0], 5]).any()


def test_window_row_that_sees_an_infinite_value_at_its_end(dev):
    """Decoded tokens whose own value is infinite in one column: a weight enters the product in three bf16 parts, all positive for about a quarter of
    the rows, and these have an infinite result.  Nothing that lies behind the last key in its tile turns it into a NaN."""
    from mini_sglang_amd import mixops

    g = torch.Generator().manual_seed(3)
    lens = [5 + 29 * b for b in range(20)]
    lens = [n + (n % 32 == 0) for n in lens]
    table, at = torch.zeros((len(lens), 600), dtype=torch.int32), 0
    for b, n in enumerate(lens):
        table[b, :n] = torch.arange(at, at + n)
        at += n
    ends = torch.tensor(lens).cumsum(0) - 1
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)  # noqa: E731
    key, value = (torch.randn(at, 512, generator=g).bfloat16() for _ in range(2))
    value[ends, 5::128] = torch.inf
    q = torch.randn(len(lens), 16 * 129, generator=g).bfloat16().to(dev)
    for splits in (1, 3):
        out = torch.empty((len(lens), 16 * 128), dtype=torch.bfloat16, device=dev)
        mixops.window_attn(out, q, 16 * 128, key.to(dev), value.to(dev), table.to(dev), i32(range(len(lens))), i32(lens), i32(range(len(lens) + 1)), len(lens),
                           16, 4, 128, 128, 0, 0.05, torch.eye(16, device=dev) + 0.1, splits=splits, max_keys=max(lens))
        hit = out[:, 5::128]
        assert not torch.isfinite(hit).any() and torch.isposinf(hit).float().mean() > 0.1
        keep = torch.ones(16 * 128, dtype=torch.bool, device=dev)
        keep[5::128] = False
        assert torch.isfinite(out[:, keep]).all()


@pytest.mark.parametrize("lens,N,K", [((1, 3, 40), 72, 64), ((64, 65, 127), 264, 96), ((256, 511, 300) * 20, 520, 64)], ids=["short", "middling", "long"])
def test_product_row_and_column_that_a_number_reaches(dev, lens, N, K):
    """Segmented products: an operand's row with a NaN or an infinity makes its row or column of the result undefined and leaves the rest its bits."""
    from mini_sglang_amd import mixops

    g = torch.Generator().manual_seed(N + K)
    E, rows = len(lens), sum(lens)
    seg = torch.tensor((0,) + lens).cumsum(0).int()
    a, b = (torch.randn(*s, K, generator=g).bfloat16().to(dev) for s in ((rows,), (E, N)))

    def product(a, b):
        c = torch.empty((rows, N), device=dev)
        mixops.gemm_nt(c, a, b, rows, N, K, lda=K, ldb=K, ldc=N, groups=E, b_gs=N * K, seg=seg.to(dev))
        return c

    clean = product(a, b)
    m, e, n = rows - 1, 1, N // 2 + 1
    for x in (torch.nan, torch.inf):
        a2, b2 = a.clone(), b.clone()
        a2[m, K - 1], b2[e, n, 1] = x, x
        got, hit = product(a2, b2), torch.zeros((rows, N), dtype=torch.bool, device=dev)
        hit[m], hit[int(seg[e]): int(seg[e + 1]), n] = True, True
        assert not torch.isfinite(got[hit]).any() and torch.equal(got[~hit], clean[~hit])

"""Small decode batches: the add + RMSNorm inside the projection's launch (msgl_skinny_norm_gemm_nt) gives the bits of the separate
launches, and the kernel with four weight rows per workgroup (msgl_skinny_quarter_gemm_nt) is the product."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops(dev):
    from mini_sglang_amd import ops as o

    return o


def _rnd(g, *shape, dtype, std=1.0):
    return (torch.randn(shape, generator=g, device=g.device) * std).to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("silu", [False, True], ids=["plain", "silu"])
@pytest.mark.parametrize("M,K", [(1, 192), (3, 256), (8, 1024), (1, 1024), (5, 960), (2, 1088), (1, 5120), (3, 2560), (1, 8192)])
def test_norm_inside_the_projection_has_the_bits_of_the_separate_launches(ops, dev, dtype, silu, M, K):
    """Fewer blocks than a wave asks for at once, one to eight rows, rows of one and of several 64-piece groups, partial groups."""
    g = torch.Generator(device=dev).manual_seed(M * 7919 + K)
    N = 192
    xb, rb = _rnd(g, M, K + 8, dtype=dtype), _rnd(g, M, K + 16, dtype=dtype)  # rows of a wider buffer
    x, res = xb[:, :K], rb[:, 8: K + 8]
    w, gamma = _rnd(g, N, K, dtype=dtype, std=K ** -0.5), _rnd(g, K, dtype=dtype)
    ran = 0
    for sl in (2, 4, 8, 16):
        for nt in (1, 2):
            if not ops.norm_linear_supported(M, N, K, sl, nt, silu):
                continue
            y, r = x.clone(), res.clone()
            ops.fused_add_rmsnorm(y, r, gamma, 1e-6)
            want = ops.skinny_linear_silu(y, w, sl, None, nt) if silu else ops.skinny_linear(y, w, sl, None, nt)
            new = torch.full((M, K + 8), 7.0, dtype=dtype, device=dev)
            out = torch.full((M + 1, want.shape[1] + 8), 7.0, dtype=dtype, device=dev)
            got = ops.norm_linear(x, w, sl, nt, res, new[:, :K], gamma, 1e-6, silu, out[:M, : want.shape[1]])
            assert torch.equal(got, want) and torch.equal(new[:, :K], r), (sl, nt)
            assert bool((new[:, K:] == 7).all()) and bool((out[M:] == 7).all()) and bool((out[:, want.shape[1]:] == 7).all())
            ran += 1
    assert ran


def test_norm_inside_the_projection_refuses_what_it_cannot_hold(ops, dev):
    x = torch.zeros((8, 1024), dtype=torch.bfloat16, device=dev)
    w, gamma, r = torch.zeros((64, 1024), dtype=torch.bfloat16, device=dev), x[0].clone(), torch.empty_like(x)
    assert not ops.norm_linear_supported(8, 64, 1024, 2, 1) and not ops.norm_linear_supported(9, 64, 1024, 16, 1)
    assert not ops.norm_linear_supported(1, 64, 128, 2, 1) and not ops.norm_linear_supported(8, 64, 8192, 16, 1)
    for slices, res_out in ((2, r), (8, x)):  # rows for more than two waves; the residual into the operand
        with pytest.raises(Exception):
            ops.norm_linear(x, w, slices, 1, x.clone(), res_out, gamma, 1e-6)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("M", [1, 3, 4, 5, 8])
@pytest.mark.parametrize("N,K", [(4, 128), (12, 256), (1024, 2048), (1028, 3072), (64, 17408), (16, 896)])
def test_four_rows_per_workgroup_is_the_product(ops, dev, dtype, M, N, K):
    g = torch.Generator(device=dev).manual_seed(M * 31 + N + K)
    x, w = _rnd(g, M, K + 8, dtype=dtype)[:, :K], _rnd(g, N, K + 8, dtype=dtype, std=K ** -0.5)[:, :K]
    want = x.double() @ w.double().t()
    eps = torch.finfo(dtype).eps
    for sl in [s for s in (1, 3, 4, 8, 16) if s <= K // 128]:
        out = torch.full((M + 1, N + 4), 7.0, dtype=dtype, device=dev)
        got = ops.skinny_linear(x, w, sl, out[:M, :N], ops.QUARTER_TILE)
        # one rounding to the 16-bit type, and K fp32 additions of products of unit size
        err = (got.double() - want).abs()
        assert bool((err <= want.abs() * eps / 2 + K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())).all()), (sl, err.max())
        assert bool((out[M:] == 7).all()) and bool((out[:, N:] == 7).all())


@pytest.mark.parametrize("M", [4, 48, 200])
def test_plan_search_times_every_family_behind_a_busy_gpu(ops, dev, monkeypatch, M):
    """The hand-written kernels' times are all taken the same way: issued from the host, every launch below 8 us measures as 8 us."""
    from mini_sglang_amd.gemm_plan import tune_projection_gemms

    clock, sleep, inside, outside = ops._time_launches_us, torch.cuda._sleep, [False], []
    timed, slept = set(), [0]

    def sleeping(cycles):
        slept[0] += 1
        return sleep(cycles)

    def recording(fn, weights, iters, rounds, *a, **k):
        inside[0], slept[0] = True, 0
        try:
            return clock(fn, weights, iters, rounds, *a, **k)
        finally:
            inside[0] = False
            assert slept[0] == rounds

    def watch(name):
        plain = getattr(ops, name)

        def call(*a, **k):
            (timed.add if inside[0] else outside.append)(name)
            return plain(*a, **k)

        monkeypatch.setattr(ops, name, call)

    families = ["skinny_linear", "skinny_linear_silu", "norm_linear", "wstream_linear", "full_batch_linear", "g3_linear", "ro_linear"]
    for name in families:
        watch(name)
    monkeypatch.setattr(ops, "_time_launches_us", recording)
    monkeypatch.setattr(torch.cuda, "_sleep", sleeping)
    g = torch.Generator(device=dev).manual_seed(M)
    N, K = 2048, 1024
    ws = [ops.interleave_gate_up(_rnd(g, N, K, dtype=torch.bfloat16, std=K ** -0.5)) for _ in range(3)]
    try:
        rep = tune_projection_gemms([("gate_up", ws, K, {"silu_interleaved": True, "fold": "norm"})], [M], "heuristic", torch.bfloat16, dev)
        want = {4: {"skinny_linear", "skinny_linear_silu", "norm_linear", "ro_linear"},
                48: {"skinny_linear", "skinny_linear_silu", "wstream_linear", "ro_linear"},
                200: {"wstream_linear", "full_batch_linear", "g3_linear", "ro_linear"}}[M]
        assert want <= timed and not outside
        r = rep[0]
        if r.get("norm_used"):  # the plan that runs is the one that is reported
            assert "norm" in r["kernel"] and r["best_us"] == r["norm_fused_us"] and r["skinny_used"]
    finally:
        ops.reset_gemm_plans()

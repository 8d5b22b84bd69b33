"""The order in which the delta rule's walks start (longest requests first, the second round of the compute units in reverse) does not
show: a batch gives every request the bits it gets alone."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,lens", [
    (16, [40, 100, 7]),                      # two requests fill the compute units once, one in the second round
    (16, [33, 16, 80, 64]),                  # two full rounds
    (16, [20, 17, 900, 5, 33, 48, 1]),       # more than two rounds, one request as long as a place's share
    (16, [30, 31, 32, 33, 34, 35, 36]),      # more than two rounds, all alike: as they come
    (8, [50, 0, 18, 70, 70, 200, 16]),       # four a round, a request without tokens, equal ones
    (3, [24] + [3, 19, 40, 11] * 16),        # more requests than lanes
])
def test_delta_walk_order(dev, monkeypatch, H, lens):
    from mini_sglang_amd import mixops

    monkeypatch.setattr(mixops, "delta_in_blocks", lambda *a, **k: True)
    d = dv = 128
    g = torch.Generator(device=dev).manual_seed(21)
    rnd = lambda *s: torch.randn(s, generator=g, device=dev)
    T, B = sum(lens), len(lens)
    qkv, b, a = rnd(T, 3 * H * d), rnd(T, H), rnd(T, H * d)
    heads = qkv[:, : 2 * H * d].view(T, 2 * H, d)
    heads /= heads.norm(dim=-1, keepdim=True)  # longer keys than 1 and the recurrence grows without end
    rate, dt, start = -torch.exp(0.1 * rnd(H)), rnd(H * d), rnd(B, H, d, dv)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)

    def call(first, last):
        n = lens[first:last]
        state, rows = start.clone(), slice(sum(lens[:first]), sum(lens[:last]))
        out = torch.empty((sum(n), H * dv), device=dev)
        cu = [sum(n[:i]) for i in range(len(n) + 1)]
        mixops.delta_rule(out, qkv[rows].contiguous(), state, b[rows], a[rows], True, rate, dt, i32(cu), i32([k + 1 for k in n]), i32(list(range(first, last))),
                          len(n), H)
        return out, state

    out, state = call(0, B)
    for r in range(B):
        if lens[r]:
            one, own = call(r, r + 1)
            assert torch.equal(out[sum(lens[:r]): sum(lens[: r + 1])], one) and torch.equal(state[r], own[r])
        else:
            assert torch.equal(state[r], start[r])

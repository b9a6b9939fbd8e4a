"""The experts' products for experts of many rows (tiles of up to 256 rows, both operands through LDS) at the edges of its
tiles, against the same sums in float64, and against the kernel for few rows, whose bits it has to give."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(rows, width, ff, gated, seed=0):
    """One choice a token: expert e gets rows[e] tokens."""
    g = torch.Generator().manual_seed(seed)
    experts, tokens = len(rows), sum(rows)
    ids = torch.cat([torch.full((n,), e, dtype=torch.int32) for e, n in enumerate(rows)])[torch.randperm(tokens, generator=g)]
    x = torch.randn((tokens, width), generator=g).bfloat16()
    up = (torch.randn((experts * ff * (2 if gated else 1), width), generator=g) * width ** -0.5).bfloat16()
    down = (torch.randn((experts * width, ff), generator=g) * ff ** -0.5).bfloat16()
    weights = torch.rand((tokens, 1), generator=g) + 0.5
    return x, ids[:, None].contiguous(), weights, up, down


def _want(x, ids, weights, up, down, experts, gated):
    width, ff = x.shape[1], down.shape[1]
    out = torch.zeros(x.shape, dtype=torch.float64)
    for e in range(experts):
        at = (ids[:, 0] == e).nonzero()[:, 0]
        h = x[at].double() @ up.view(experts, -1, width)[e].double().T
        h = torch.nn.functional.silu(h[:, :ff]) * h[:, ff:] if gated else torch.relu(h).square()
        out[at] = weights[at].double() * (h.bfloat16().double() @ down.view(experts, width, ff)[e].double().T)
    return out


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("rows,width,ff", [
    ([255, 256, 257, 1], 64, 64),             # one stage of columns; a tile's last row, its end, a second tile
    ([63, 64, 65, 129, 193], 192, 128),       # the number of blocks of 16 rows a wave multiplies
    ([0, 700, 0, 3], 128, 320),               # experts without a token; outputs that end inside a tile
    ([40, 41], 576, 192)])
def test_experts_of_many_rows(rows, width, ff, gated):
    from nano_vllm_amd.kernels import HipKernels
    k = HipKernels(DEV, torch.bfloat16, quiet=True)
    x, ids, weights, up, down = _case(rows, width, ff, gated)
    act = "silu" if gated else "relu2"
    run = lambda t: k.moe_experts(t[0], t[1], t[2], up.to(DEV), down.to(DEV), len(rows), act, gated=gated)
    got = run([t.to(DEV) for t in (x, ids, weights)])
    want = _want(x, ids, weights, up, down, len(rows), gated)
    # the inner layer is rounded by both (an entry whose sum lies at a rounding edge may fall either way), the result once more
    err = (got.double().cpu() - want).abs()
    assert float(err.max()) <= 2 ** -7 * float(want.abs().max()), float(err.max() / want.abs().max())
    # a handful of tokens alone takes the tiles of 32 rows: a token's result must not depend on what else is in the batch
    few = torch.randperm(x.shape[0], generator=torch.Generator().manual_seed(1))[:5]
    alone = run([t[few].contiguous().to(DEV) for t in (x, ids, weights)])
    assert torch.equal(alone, got[few.to(DEV)])


def test_rows_that_are_not_aligned():
    """Columns of wider rows at an odd offset: no vector loads, tiles of 32 rows, the same sums."""
    from nano_vllm_amd.kernels import HipKernels
    k = HipKernels(DEV, torch.bfloat16, quiet=True)
    x, ids, weights, up, down = _case([300, 40, 100], 128, 64, True)
    wide = torch.zeros((x.shape[0], 131), dtype=torch.bfloat16)
    wide[:, 1:129] = x
    got = k.moe_experts(wide.to(DEV)[:, 1:129], ids.to(DEV), weights.to(DEV), up.to(DEV), down.to(DEV), 3, "silu", gated=True)
    want = _want(x, ids, weights, up, down, 3, True)
    assert float((got.double().cpu() - want).abs().max()) <= 2 ** -7 * float(want.abs().max())


@pytest.mark.parametrize("routing", ["sigmoid_groups", "softmax_top", "softmax_choice", "softmax_scores"])
@pytest.mark.parametrize("experts,groups,keep,top", [(64, 1, 1, 8), (64, 8, 3, 24), (32, 4, 2, 8), (63, 21, 5, 3), (6, 6, 2, 2), (1, 1, 1, 1), (64, 64, 64, 64)])
def test_routing_with_an_expert_a_lane(routing, experts, groups, keep, top):
    """Up to 64 experts and more run kernels of their own: groups of experts that nobody chooses beside them change no bit.
    Many scores are equal (the lower number goes first)."""
    from nano_vllm_amd.kernels import HipKernels
    k = HipKernels(DEV, torch.bfloat16, quiet=True)
    g = torch.Generator().manual_seed(experts + top)
    logits = (torch.randn((37, experts), generator=g) * 4).round() / 2
    bias = (torch.randn(experts, generator=g) * 2).round() / 8 if routing in ("softmax_top", "softmax_choice") else None
    if routing == "softmax_top":
        groups = keep = 1
    per = experts // groups
    more = (64 // per + 1) * per
    wide = torch.cat((logits, torch.full((37, more), float("-inf"))), 1)
    wide_bias = None if bias is None else torch.cat((bias, torch.full((more,), -9.0)))
    dev = lambda t: None if t is None else t.to(DEV)
    one = k.moe_route(dev(logits), top, groups, keep, 1.7, routing=routing, bias=dev(bias))
    two = k.moe_route(dev(wide), top, groups + more // per, keep, 1.7, routing=routing, bias=dev(wide_bias)) if routing != "softmax_top" else \
        k.moe_route(dev(wide), top, 1, 1, 1.7, routing=routing, bias=dev(wide_bias))
    assert torch.equal(one[0], two[0]) and torch.equal(one[1], two[1])
    assert int(one[0].max()) < experts and all(len(set(r)) == top for r in one[0].tolist())


@pytest.mark.parametrize("tokens", [2047, 2048, 2049])
def test_more_pairs_than_the_plan_keeps(tokens):
    """8 choices of a token: 16384 pairs are what the plan's workgroup keeps in registers."""
    from nano_vllm_amd.kernels import HipKernels
    k = HipKernels(DEV, torch.bfloat16, quiet=True)
    g = torch.Generator().manual_seed(tokens)
    x, up, down = (torch.randn(s, generator=g).bfloat16().to(DEV) for s in ((tokens, 64), (10 * 64, 64), (10 * 64, 64)))
    ids = torch.rand((tokens, 12), generator=g).topk(8, 1)[1].int().to(DEV)         # (10 and 11: identities)
    weights = torch.rand((tokens, 8), generator=g).to(DEV)
    run = lambda a, b: k.moe_experts(x[a:b], ids[a:b].contiguous(), weights[a:b].contiguous(), up, down, 10)
    assert torch.equal(run(0, tokens), torch.cat((run(0, 1000), run(1000, tokens))))

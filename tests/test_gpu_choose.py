"""Experts chosen from router logits that another product formed (skyrl_moe_choose, and the choice of up to 64 experts inside
skyrl_moe_route) against the oracle's routing of the same f32 scores, and a step's product and choice against the router's own
launches."""

import pytest
import torch

from oracle import hybrid_ref
from skyrl_amd.inference_engines import layer_kernels as lk

pytestmark = pytest.mark.gpu


def _pairs(idx, order, tile_expert, tm):
    """{pair: expert} that the tiles list."""
    out = {}
    for tile, e in enumerate(tile_expert[:-1].tolist()):
        for p in order[tile].tolist() if e >= 0 else ():
            if p >= 0:
                assert p not in out
                out[p] = e
    assert sum(e >= 0 for e in tile_expert[:-1].tolist()) == int(tile_expert[-1])
    return out


# groups of powers of two and others, one group, one expert per group, all kept, all experts chosen; rows on both sides of
# what one launch sorts
@pytest.mark.parametrize("experts,groups,keep,top", [(64, 8, 4, 8), (64, 1, 1, 6), (60, 12, 5, 7), (64, 32, 9, 8), (64, 16, 5, 8),
                                                     (64, 4, 2, 8), (64, 2, 1, 8), (64, 64, 20, 8), (16, 16, 3, 3), (33, 3, 2, 22),
                                                     (8, 2, 2, 8), (1, 1, 1, 1)])
@pytest.mark.parametrize("n,shares", [(1, 1), (5, 3), (16, 2), (46, 8), (129, 2)])
def test_choice(dev, experts, groups, keep, top, n, shares):
    g = torch.Generator(device=dev).manual_seed(experts + n)
    sh = lk.moe_shape(64, 64, experts, top, groups, keep)
    logits = torch.randn(shares, n, 24 + experts, device=dev, generator=g)
    corr = torch.randn(experts, device=dev, generator=g) * 0.3
    tm = 16
    idx, weight, order, tile_expert = lk.moe_choose(sh, logits, 24, corr, tm)
    z = logits[0, :, 24:].clone()
    for i in range(1, shares):
        z += logits[i, :, 24:]
    scores = torch.sigmoid(z.double()).cpu()
    want, _ = hybrid_ref.route(scores, corr.double().cpu(), top, groups, keep)
    chosen = lambda i: (scores + corr.double().cpu()).gather(1, i.cpu().long())  # noqa: E731
    assert bool((idx.sort(1).values[:, 1:] != idx.sort(1).values[:, :-1]).all()) and bool(((idx >= 0) & (idx < experts)).all())
    # equal but for places that f32 scores cannot tell apart
    torch.testing.assert_close(chosen(idx), chosen(want), atol=3e-7, rtol=0)
    torch.testing.assert_close(weight.double().cpu(), scores.gather(1, idx.cpu().long()), atol=3e-7, rtol=0)
    assert _pairs(idx, order, tile_expert, tm) == {t * top + k: e for t, row in enumerate(idx.tolist()) for k, e in enumerate(row)}


def test_ties_and_what_is_no_number(dev):
    sh = lk.moe_shape(64, 64, 64, 8, 8, 4)
    corr = torch.zeros(64, device=dev)
    z = torch.zeros(1, 3, 64, device=dev)
    z[0, 1] = float("nan")
    z[0, 2, 40:48] = float("inf")
    idx, weight, order, tile_expert = lk.moe_choose(sh, z, 0, corr, 16)
    assert idx[0].tolist() == list(range(8))  # the lower expert first
    assert 0 <= int(idx[1].min()) and int(idx[1].max()) < 64
    assert idx[2].tolist() == list(range(40, 48)) and weight[2].tolist() == [1.0] * 8
    assert len(_pairs(idx, order, tile_expert, 16)) == 24


@pytest.mark.parametrize("n", (1, 17, 64, 128))
def test_joint_product_chooses_as_the_router(dev, n):
    g = torch.Generator(device=dev).manual_seed(n)
    sh = lk.moe_shape(512, 64, 64, 8, 8, 4)
    joint = (torch.randn(512 + 64, 512, device=dev, generator=g) * 0.05).bfloat16()
    x = torch.randn(n, 512, device=dev, generator=g).bfloat16()
    corr = torch.randn(64, device=dev, generator=g) * 0.1
    idx, weight, _, _ = lk.moe_choose(sh, lk.linear(x, joint, parts=True), 512, corr, 16)
    other, w2 = lk.moe_route(sh, x, joint[512:].contiguous(), corr)
    at = torch.sigmoid(x.double() @ joint[512:].double().t())
    pick = lambda i: (at + corr.double()).gather(1, i.long())  # noqa: E731
    torch.testing.assert_close(pick(idx), pick(other), atol=1e-5, rtol=0)
    torch.testing.assert_close(weight.double(), at.gather(1, idx.long()), atol=1e-5, rtol=0)


@pytest.mark.parametrize("experts,groups,keep,top,width,ff", [(64, 8, 4, 8, 512, 96), (60, 12, 5, 7, 72, 40), (33, 3, 2, 22, 64, 8),
                                                              (8, 2, 2, 8, 2048, 768), (1, 1, 1, 1, 8, 24)])
@pytest.mark.parametrize("shares", (1, 3))
def test_choice_in_the_first_product(dev, experts, groups, keep, top, width, ff, shares):
    """One token: the experts and weights of moe_choose and, bit for bit, the rows of its products."""
    g = torch.Generator(device=dev).manual_seed(experts + shares)
    sh = lk.moe_shape(width, ff, experts, top, groups, keep)
    logits = torch.randn(shares, 1, 24 + experts, device=dev, generator=g)
    corr = torch.randn(experts, device=dev, generator=g) * 0.3
    rand = lambda *s: (torch.randn(*s, device=dev, generator=g) * 0.1).bfloat16()  # noqa: E731
    x, gate_up, down = rand(1, width), rand(experts, 2, ff, width), rand(experts, width, ff)
    for z in (logits, torch.full_like(logits, float("nan"))):
        idx, weight, order, tile_expert = lk.moe_choose(sh, z, 24, corr, 16)
        want = lk.moe_experts(sh, x, idx, weight, gate_up, down, 16, (order, tile_expert))
        got = lk.moe_one(sh, z, 24, corr, x, gate_up, down)
        if z is logits:
            assert torch.equal(got, want) and got.shape == (top, width)
        else:
            assert bool(got.isnan().all())
    assert lk.moe_one(sh, logits, 24, corr, torch.cat([x, x]), gate_up, down) is None

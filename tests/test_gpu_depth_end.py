"""pta_depth_end against the four entry points that it does in one launch: launch after launch with one workspace, and recorded in a graph."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# rows, width, features of the token's own part, depths, parts (0: none), experts (0: no routing): one block and one tile, remainders of both, the most of each,
# widths that are no multiple of eight, of four and of two
SHAPES = [(2, 76, 16, 2, 2, 3), (1, 70, 8, 1, 0, 0), (3, 70, 24, 3, 2, 5), (2, 1001, 136, 2, 1, 0), (4, 8190, 1024, 3, 2, 4), (1, 72, 8, 1, 0, 0), (2, 2048, 256, 3, 3, 0), (1, 2056, 264, 9, 2, 5), (4, 4096, 256, 2, 3, 8), (3, 1000, 136, 4, 0, 4), (4, 8192, 1024, 2, 2, 0), (4, 136, 24, 3, 1, 0)]


@pytest.mark.parametrize("rows, width, side, depths, n_parts, experts", SHAPES)
def test_as_the_four_calls(rows, width, side, depths, n_parts, experts):
    from poptransformer_amd import _hybrid_lib as H
    from poptransformer_amd import hybrid_kernels as HK
    g = torch.Generator(device="cuda").manual_seed(71)

    def f32(*shape, scale=1.0):
        return torch.randn(shape, generator=g, device="cuda") * scale
    ld = HK.pad8(width)
    gate, proj = HK.WideWeight(f32(side, width, scale=width ** -0.5), torch.bfloat16), HK.WideWeight(f32(width, side, scale=side ** -0.5), torch.bfloat16)
    history, h_one = f32(depths + 1, (rows + 3) // 4 * 4, width), torch.zeros((rows, ld), dtype=torch.bfloat16, device="cuda")
    rounded, act, y = torch.zeros_like(h_one), torch.zeros((rows, side), dtype=torch.bfloat16, device="cuda"), f32(rows, width)
    y_weight, norm_weight, weights = f32(width), f32(width), f32(depths)
    router = f32(experts, ld).bfloat16() if experts else None
    routing = [HK.Routing(rows, experts, 2, False, 1.0, "cuda", H.SCORE_SOFTMAX, 1, 1, False) for _ in (0, 1)] if experts else [None, None]
    workspace = HK.depth_end_workspace(rows, width, side, torch.bfloat16, "cuda")
    one, x_one = history.clone(), None
    h, parts, weight, own = torch.zeros_like(h_one), f32(rows, max(n_parts, 1), width), f32(rows, max(n_parts, 1)), f32(rows, side).bfloat16()

    def keywords(i):
        return dict(rows=rows, eps=1e-5, h=(h_one, h)[i], norm_weight=norm_weight, weights=weights, y_weight=y_weight, next=depths,
                    **(dict(router=router, routing=routing[i]) if experts else {}))
    added = dict(parts=parts, n_parts=n_parts, part_weight=weight) if n_parts else {}

    def launch():
        HK.depth_end(history[depths - 1], rows, rounded, added, gate, own, proj, (history, depths, keywords(1)), workspace)

    def again(k):
        """other values in the same places, the four calls, and the bound on what they may differ by"""
        for t in (history, parts, weight):
            t.normal_(generator=g)
        own.copy_(f32(rows, side))
        one.copy_(history)
        HK.add_parts(one[depths - 1], rows, rounded, **added)
        HK.linear(rounded, gate, act, rows, act=H.ACT_GELU_TANH, mul=own)
        HK.linear(act, proj, y, rows, ld=width)
        x = one[depths - 1].clone()
        HK.depth_norm(one, depths, y=y, **keywords(0))
        # The gate's fp32 sums may round to the other neighbour of bf16 (2^-8): in y that, its sums' order and what that does to its norm
        dy = (act.double().abs() @ proj_plain.abs().T) * (2.0 ** -8 + side * 2.0 ** -23)
        inv = 1.0 / (y.double().pow(2).mean(1, keepdim=True) + 1e-5).sqrt()
        dv = (dy + y.double().abs() * dy.pow(2).mean(1, keepdim=True).sqrt() * inv) * inv * y_weight.double().abs() + 2.0 ** -22 * (one[depths - 1][:rows].double().abs() + x[:rows].double().abs())
        du = dv * weights[-1].double().abs() + 2.0 ** -21 * (1 + one[depths][:rows].double().abs())
        u = one[depths][:rows].double()
        f = 1.0 / (u.var(1, unbiased=False, keepdim=True) + 1e-5).sqrt()
        move = du.pow(2).mean(1, keepdim=True).sqrt()                            # of the mean and of the root mean square, at most
        dh = (du + move + (u - u.mean(1, keepdim=True)).abs() * move * f) * f * norm_weight.double().abs() + 2.0 ** -7 * h_one[:, :width].double().abs()
        return dv, du, dh

    from poptransformer_amd import kernels  # noqa: F401
    w = torch.zeros((width, side), dtype=torch.float64, device="cuda")
    g2 = torch.Generator(device="cuda").manual_seed(71)
    torch.randn((side, width), generator=g2, device="cuda")
    w.copy_((torch.randn((width, side), generator=g2, device="cuda") * side ** -0.5).bfloat16())
    proj_plain = w

    def check(bounds):
        dv, du, dh = bounds
        for got, ref, bound in ((history[depths - 1], one[depths - 1], dv), (history[depths], one[depths], du), (h, h_one, dh)):
            cols = slice(0, width)
            d = (got[:rows, cols].double() - ref[:rows, cols].double()).abs()
            assert (d <= bound).all(), (d / bound).max().item()
        assert torch.equal(h[:, width:], h_one[:, width:])
        if experts:
            assert torch.allclose(routing[0].weights, routing[1].weights, rtol=0.1, atol=0.02)

    for k in range(3):
        bounds = again(k)
        launch()
        check(bounds)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        launch()
    for k in range(3):
        bounds = again(k)
        graph.replay()
        check(bounds)
        torch.cuda.synchronize()
    assert not torch.isnan(h).any()


@pytest.mark.parametrize("width, h_ld", [(12, 13), (64, 71), (1000, 1002), (70, 70)])
def test_rows_of_h_that_are_not_whole_pieces(width, h_ld):
    """h may have any number of columns from the width to seven more."""
    from poptransformer_amd import hybrid_kernels as HK
    g = torch.Generator(device="cuda").manual_seed(5)

    def f32(*shape):
        return torch.randn(shape, generator=g, device="cuda")
    side, rows, bf16 = 24, 3, torch.bfloat16
    gate, proj = HK.WideWeight(f32(side, width), bf16), HK.WideWeight(f32(width, side), bf16)
    x, rounded, own = f32(3, 4, width), torch.zeros(rows, HK.pad8(width), dtype=bf16, device="cuda"), f32(rows, side).bfloat16()
    ws, results = HK.depth_end_workspace(rows, width, side, bf16, "cuda"), []
    kw = dict(rows=rows, eps=1e-5, norm_weight=f32(width), weights=f32(2), y_weight=f32(width), next=2)
    for ld in (HK.pad8(width), h_ld):
        history, h = x.clone(), torch.full((rows + 1, ld), 7.0, dtype=bf16, device="cuda")
        HK.depth_end(history[1], rows, rounded, {}, gate, own, proj, (history, 2, dict(kw, h=h)), ws)
        assert (h[:rows, width:] == 0).all() and (h[rows] == 7).all()
        results.append((history, h[:rows, :width].float()))
    (ha, a), (hb, b) = results
    # (sums of whole pieces and of single columns in another order: fp32, then to one or the other neighbour of bf16)
    assert torch.allclose(ha, hb, rtol=1e-5, atol=1e-5) and ((a - b).abs() <= 2.0 ** -7 * a.abs() + 1e-4).all()


def test_what_is_refused():
    from poptransformer_amd import hybrid_kernels as HK
    for rows, width, side, dtype in ((5, 2048, 256, torch.bfloat16), (1, 8200, 256, torch.bfloat16), (1, 2048, 1032, torch.bfloat16), (1, 2048, 256, torch.float32)):
        assert HK.depth_end_workspace(rows, width, side, dtype, "cuda") is None
    gate, proj = HK.WideWeight(torch.randn(24, 64, device="cuda"), torch.bfloat16), HK.WideWeight(torch.randn(64, 24, device="cuda"), torch.bfloat16)
    x, h, own = torch.randn(2, 1, 64, device="cuda"), torch.zeros(1, 64, dtype=torch.bfloat16, device="cuda"), torch.randn(1, 24, device="cuda").bfloat16()
    kw = dict(rows=1, eps=1e-5, h=h, norm_weight=torch.ones(64, device="cuda"), weights=torch.ones(1, device="cuda"), y_weight=torch.ones(64, device="cuda"))
    ws = HK.depth_end_workspace(1, 64, 24, torch.bfloat16, "cuda")
    with pytest.raises(ValueError):                                              # the wrong weight
        HK.depth_end(x[0], 1, h, {}, proj, own, gate, (x, 1, kw), ws)
    with pytest.raises(ValueError):                                              # a workspace of too few bytes
        HK.depth_end(x[0], 1, h, {}, gate, own, proj, (x, 1, kw), ws[:-64])
    with pytest.raises(ValueError):                                              # not the newest depth
        HK.depth_end(x[1], 1, h, {}, gate, own, proj, (x, 1, kw), ws)


def test_a_wait_that_gave_up_leaves_no_numbers():
    """The word that a wait sets when it gives up, set by hand: every launch ends, and h is NaN."""
    from poptransformer_amd import hybrid_kernels as HK
    gate, proj = HK.WideWeight(torch.randn(24, 64, device="cuda"), torch.bfloat16), HK.WideWeight(torch.randn(64, 24, device="cuda"), torch.bfloat16)
    x, h, own = torch.randn(1, 4, 64, device="cuda"), torch.zeros(2, 64, dtype=torch.bfloat16, device="cuda"), torch.randn(2, 24, device="cuda").bfloat16()
    kw = dict(rows=2, eps=1e-5, h=h, norm_weight=torch.ones(64, device="cuda"), weights=torch.ones(1, device="cuda"), y_weight=torch.ones(64, device="cuda"))
    ws = HK.depth_end_workspace(2, 64, 24, torch.bfloat16, "cuda")
    for failed in (0, 1, 1):
        ws.view(torch.int32)[2] = failed
        HK.depth_end(x[0], 2, h, {}, gate, own, proj, (x, 1, kw), ws)
        assert bool(torch.isnan(h.float()).all()) == bool(failed) and (failed or not torch.isnan(h.float()).any())

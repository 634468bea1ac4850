"""pta_linear_then_norm against pta_linear and the norm's own entry point, bit for bit: products whose K is split (the slices are added and the rows
normed by one launch) and products whose K is not."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def weight(kind, N, Kd, g):
    from poptransformer_amd import kernels as K
    w = torch.randn((N, Kd), generator=g, device="cuda") * 0.05
    if kind == "f16":
        return K.F16Weight(w.half())
    if kind == "int4":
        return K.W4Weight(torch.randint(-128, 128, (N, Kd // 2), generator=g, device="cuda").to(torch.int8), (torch.rand(N, generator=g, device="cuda") * 0.01).half())
    scale = torch.tensor([-1], dtype=torch.int32, device="cuda")
    return K.F8Weight(K.half_to_fp8(w.half(), scale, kind), scale, kind)


# rows, features, channels, whether K is split where there is a workspace: the fewest and the most columns of a row, rows one past a tile, no split
SHAPES = {"int4": [(32, 16384, 4096, True), (17, 8192, 8, None), (257, 8192, 2048, None), (1000, 11008, 4096, True), (20, 256, 4096, False)],
          "f16": [(33, 8192, 1032, None), (300, 4104, 1024, None), (129, 16384, 8184, None), (5, 4096, 4096, False)],
          "F143": [(1020, 13704, 4096, True), (40, 13696, 4096, None), (200, 4096, 2048, None)],
          "F152": [(64, 8192, 2056, None)]}


@pytest.mark.parametrize("kind, M, Kd, N, split", [(k, *s) for k, shapes in SHAPES.items() for s in shapes])
@pytest.mark.parametrize("form", ["rms", "grid", "layer", "shift"])
def test_as_the_two_calls(kind, M, Kd, N, split, form):
    from poptransformer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(61)
    x = torch.randn((M, Kd), generator=g, device="cuda").half() * 0.1
    w = weight(kind, N, Kd, g)

    def rows(*shape):
        return torch.randn(shape, generator=g, device="cuda").half()
    gamma, beta, bias, mul, res, prev = rows(N), rows(N), rows(N), rows(M, N), rows(M, N), rows(M, N)
    mixes, exponent = [rows(N) for _ in range(3)], torch.tensor([-2], dtype=torch.int32, device="cuda")
    ends = {"rms": dict(residual=res), "grid": dict(bias=bias, residual=res), "layer": dict(bias=bias), "shift": dict(mul=mul, residual=res, post_scale=0.5)}[form]
    got, ref, out, one = (torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda") for _ in range(4))
    mixed, plain, before = [torch.empty_like(got) for _ in range(3)], [torch.empty_like(got) for _ in range(3)], prev.clone()
    workspace = K.linear_workspace(M, N, "cuda")
    workspace.fill_(0xFF)
    then = {"rms": lambda: K.RowNorm(gamma, None, 1e-5, out=out), "grid": lambda: K.RowNorm(gamma, None, 1e-5, out=out, grid=(exponent, "F143")),
            "layer": lambda: K.RowNorm(gamma, beta, 1e-5, out=out), "shift": lambda: K.RowNorm(gamma, beta, 1e-5, out=out, shift=(prev, mixes[:2], mixed[:2]))}[form]()
    K.linear_then_norm(x, w, got, then, workspace=workspace, **ends)
    if split is not None:
        assert split == (not torch.equal(workspace, torch.full_like(workspace, 0xFF)))
    K.linear(x, [w], [ref], workspace=workspace, **ends)
    if form == "rms":
        K.rmsnorm(ref, gamma, 1e-5, one)
    elif form == "grid":
        K.rmsnorm_fp8_grid(ref, gamma, 1e-5, exponent, "F143", out=one)
    elif form == "layer":
        K.layer_norm_ce(ref, gamma, beta, 1e-5, one)
    else:
        K.layer_norm_ce_mix(ref, gamma, beta, 1e-5, before, mixes[:2], plain[:2], out=one)
        assert torch.equal(prev, before) and all(torch.equal(a, b) for a, b in zip(mixed[:2], plain[:2]))
    assert not torch.isnan(got).any() and torch.equal(got, ref) and torch.equal(out, one)


def test_what_is_refused():
    from poptransformer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(3)
    x, w = torch.randn((20, 256), generator=g, device="cuda").half(), weight("f16", 64, 256, g)
    out, gamma = torch.empty((20, 64), dtype=torch.float16, device="cuda"), torch.ones(64, dtype=torch.float16, device="cuda")
    with pytest.raises(ValueError):
        K.linear_then_norm(x, w, out, K.RowNorm(gamma[:56].contiguous(), None, 1e-5, out=torch.empty_like(out)))
    with pytest.raises(ValueError):
        K.linear_then_norm(x, w, out, K.RowNorm(gamma, None, 1e-5, out=torch.empty((19, 64), dtype=torch.float16, device="cuda")))
    with pytest.raises(ValueError):
        K.linear_then_norm(x, w, out, K.RowNorm(gamma, None, 1e-5))
    with pytest.raises(ValueError):
        K.linear_then_norm(x, w, out, K.RowNorm(gamma, gamma, 1e-5, out=torch.empty_like(out), grid=(torch.zeros(1, dtype=torch.int32, device="cuda"), "F143")))


def test_tensors_that_the_norms_own_entry_points_refuse():
    """The result that is normed, the previous rows and the mixing vectors: as layer_norm_ce_mix and rmsnorm look at them."""
    from poptransformer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(3)
    x, w = torch.randn((20, 256), generator=g, device="cuda").half(), weight("f16", 64, 256, g)

    def rows(*shape, dtype=torch.float16):
        return torch.zeros(shape, dtype=dtype, device="cuda")
    gamma = rows(64)
    for out in (rows(20, 64, dtype=torch.float32), rows(20, 128)[:, ::2], rows(10, 128), rows(21, 64)):
        with pytest.raises(ValueError):
            K.linear_then_norm(x, w, out, K.RowNorm(gamma, None, 1e-5, out=rows(20, 64)))
    for prev, mixes, mixed in ((rows(40, 32), [gamma], [rows(20, 64)]), (rows(20, 64), [gamma, gamma], [rows(20, 64)]), (rows(20, 64), [], []),
                               (rows(20, 64), [gamma], [rows(20, 63)]), (rows(20, 64), [gamma.float()], [rows(20, 64)])):
        with pytest.raises(ValueError):
            K.linear_then_norm(x, w, rows(20, 64), K.RowNorm(gamma, gamma, 1e-5, shift=(prev, mixes, mixed)))
    with pytest.raises(ValueError):
        K.RowNorm(gamma, None, 1e-5, out=rows(20, 64), grid=(torch.zeros(1, dtype=torch.int64, device="cuda"), "F143"))
    with pytest.raises(ValueError):
        K.RowNorm(gamma.reshape(8, 8), None, 1e-5, out=rows(20, 64))


# rows, features, channels; the slices of K without and with any_order: the fewest and the most rows, more or fewer slices with it and the same, blocks of channels and feature
# tiles that do not divide
ANY_ORDER = [("int4", 12, 11008, 2048, 1, 1), ("int4", 13, 11008, 2048, 1, 4), ("int4", 16, 1024, 64, 1, 1), ("int4", 20, 11008, 4096, 2, 2), ("int4", 64, 4104, 4096, 1, 2), ("int4", 100, 16392, 2048, 4, 4),
             ("int4", 128, 3072, 768, 1, 3), ("int4", 129, 3072, 768, 1, 1), ("F143", 8, 13704, 4096, 1, 1), ("F143", 9, 13704, 4096, 1, 2), ("F143", 16, 11008, 1032, 1, 3), ("F143", 17, 8192, 2056, 3, 4),
             ("F143", 40, 4096, 4104, 2, 2), ("F143", 64, 13696, 4096, 2, 4), ("f16", 12, 16392, 2040, 1, 4), ("f16", 24, 11008, 4096, 1, 2), ("f16", 31, 2824, 1016, 1, 2), ("f16", 60, 6144, 3080, 2, 2),
             ("f16", 80, 5632, 2048, 1, 2), ("F152", 33, 4096, 1024, 2, 4), ("F152", 24, 8904, 1584, 2, 2), ("F152", 17, 5632, 3072, 1, 1),
             # a slice's groups by eights: 84 blocks in three slices are two rounds
             ("F143", 33, 6144, 1336, 2, 2), ("f16", 33, 6144, 1336, 3, 2), ("f16", 128, 8904, 3584, 1, 1)]


@pytest.mark.parametrize("kind, M, Kd, N, alone, any_order", ANY_ORDER)
@pytest.mark.parametrize("form", ["rms", "grid", "layer", "shift"])
def test_sums_in_any_order(kind, M, Kd, N, alone, any_order, form):
    """With any_order the product is cut otherwise where that is faster, and by the scratch that there is: within the bound of fp32 sums, and the norm is that of the rows it
    leaves."""
    from poptransformer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(71)
    x, w = torch.randn((M, Kd), generator=g, device="cuda").half() * 0.1, weight(kind, N, Kd, g)

    def rows(*shape):
        return torch.randn(shape, generator=g, device="cuda").half()
    gamma, beta, bias, mul, res, prev = rows(N), rows(N), rows(N), rows(M, N), rows(M, N), rows(M, N)
    mixes, exponent = [rows(N) for _ in range(3)], torch.tensor([-2], dtype=torch.int32, device="cuda")
    ends = {"rms": dict(residual=res), "grid": dict(bias=bias, residual=res), "layer": dict(bias=bias), "shift": dict(mul=mul, residual=res, post_scale=0.5)}[form]
    unit = torch.eye(Kd, dtype=torch.float16, device="cuda")
    dense = torch.cat([K.linear(unit[i:i + 256], [w], [torch.empty((min(256, Kd - i), N), dtype=torch.float16, device="cuda")])[0] for i in range(0, Kd, 256)]).double()
    ref = x.double() @ dense
    # fp32 sums of exact products within K 2^-24 of the sum of magnitudes, and fp16 roundings of the product and of each value on the way to the end: every one within
    # 2^-11 of what it rounds, which the factors behind it carry on
    err = 2.0 ** -11 * ref.abs() + (Kd + 2) * 2.0 ** -24 * (x.double().abs() @ dense.abs()) + 2.0 ** -24
    for name, t in ends.items():
        if name == "post_scale":
            ref, err = ref * t, err * t
        elif name == "mul":
            ref, err = ref * t.double(), err * t.double().abs()
        else:
            ref = ref + t.double()
        err = err + 2.0 ** -11 * (ref.abs() + err) + 2.0 ** -24
    for room in (0, 1, 2, 3, 4):
        got, out, one = (torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda") for _ in range(3))
        mixed, plain, was, before = [torch.empty_like(got) for _ in range(3)], [torch.empty_like(got) for _ in range(3)], prev.clone(), prev.clone()
        then = {"rms": dict(out=out), "grid": dict(out=out, grid=(exponent, "F143")), "layer": dict(out=out), "shift": dict(shift=(was, mixes[:2], mixed[:2]), out=out)}[form]
        workspace = K.linear_workspace(M, N, "cuda")[:room * M * N * 4] if room else None
        norm_beta = beta if form in ("layer", "shift") else None
        K.linear_then_norm(x, w, got, K.RowNorm(gamma, norm_beta, 1e-5, any_order=True, **then), workspace=workspace, **ends)
        slices = K.linear_slices()
        assert slices == any_order if room == 4 else slices <= max(room, 1)
        assert ((got.double() - ref).abs() <= err).all()
        if form == "rms":
            K.rmsnorm(got, gamma, 1e-5, one)
        elif form == "grid":
            K.rmsnorm_fp8_grid(got, gamma, 1e-5, exponent, "F143", out=one)
        elif form == "layer":
            K.layer_norm_ce(got, gamma, beta, 1e-5, one)
        else:
            K.layer_norm_ce_mix(got, gamma, beta, 1e-5, before, mixes[:2], plain[:2], out=one)
            assert torch.equal(was, before) and all(torch.equal(a, b) for a, b in zip(mixed[:2], plain[:2]))
        assert torch.equal(out, one)
    K.linear_then_norm(x, w, got, K.RowNorm(gamma, norm_beta, 1e-5, **dict(then, **({"shift": (prev.clone(), mixes[:2], mixed[:2])} if form == "shift" else {}))), workspace=workspace, **ends)
    assert K.linear_slices() == alone

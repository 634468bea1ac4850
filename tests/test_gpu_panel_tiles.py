"""Products of 33 rows and more by INT4 and F152 weights (gemm_panel_kernel) against float64: every tile of 48 to 128 rows with one, two and four parts of K, for a pair
and for others, and tiles of two kinds in one product; slices of K across workgroups; channels and features of any number.  Which tile and how many slices a launch takes
is its plan's choice, so each is asked for by sizes and looked at."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def weight(kind, N, Kd, g):
    """The weight and its values, [N, K]."""
    from poptransformer_amd import kernels as K
    if kind == "int4":
        packed = torch.randint(-128, 128, (N, Kd // 2), generator=g, device="cuda").to(torch.int8)
        scale = (torch.rand(N, generator=g, device="cuda") * 0.01).half()
        return K.W4Weight(packed, scale), K.int4_to_half(packed, scale).T.double()
    scale = torch.tensor([-1], dtype=torch.int32, device="cuda")
    codes = K.half_to_fp8((torch.randn((N, Kd), generator=g, device="cuda") * 0.05).half(), scale, "F152")
    return K.F8Weight(codes, scale, "F152"), K.fp8_to_half(codes, scale, "F152").double()


# tile (rows x channels of a workgroup: 512 channels are one part of K, 256 two, 128 four), form, rows, features, channels
TILES = {"int4": [("128x512", "three", 452, 712, 8848), ("128x512", "pair", 674, 720, 9332), ("112x512", "three", 433, 680, 8712), ("112x512", "pair", 780, 680, 7778), ("96x512", "three", 561, 680, 5504), ("96x512", "pair", 575, 680, 8456),
                  ("80x512", "three", 133, 704, 5831), ("80x512", "pair", 201, 696, 8237), ("128x256", "three", 228, 984, 7352), ("128x256", "pair", 351, 904, 8712), ("112x256", "three", 201, 912, 7320), ("112x256", "pair", 394, 936, 6978),
                  ("96x256", "three", 161, 960, 7336), ("96x256", "pair", 321, 912, 6904), ("80x256", "three", 138, 920, 7424), ("80x256", "pair", 197, 984, 8212), ("64x256", "three", 145, 912, 3680), ("64x256", "pair", 135, 904, 5912),
                  ("80x128", "three", 66, 2280, 5480), ("80x128", "pair", 68, 2144, 8649), ("64x128", "three", 99, 2064, 3591), ("64x128", "pair", 99, 2136, 5810), ("48x128", "three", 67, 2112, 2737), ("48x128", "pair", 76, 2080, 4304),
                  ("96x512 64x256", "pair", 833, 920, 9264), ("80x512 80x256", "three", 514, 912, 8770), ("112x512 80x256", "one", 1864, 1024, 9824), ("64x256", "one", 1024, 1024, 4096), ("48x128", "pair", 48, 4104, 11008)],
         "F152": [("112x512", "three", 328, 696, 7440), ("112x512", "pair", 967, 680, 4896), ("96x512", "three", 167, 728, 9272), ("96x512", "pair", 562, 760, 6188), ("80x512", "three", 131, 696, 2808), ("80x512", "pair", 141, 688, 2782),
                  ("112x256", "three", 328, 936, 3960), ("112x256", "pair", 322, 912, 6016), ("96x256", "three", 176, 904, 7234), ("96x256", "pair", 324, 928, 5608), ("80x256", "three", 129, 944, 5088), ("80x256", "pair", 134, 1016, 7524),
                  ("64x256", "three", 134, 1064, 1352), ("64x256", "pair", 130, 1128, 1454), ("80x128", "three", 130, 1944, 3600), ("80x128", "pair", 194, 1952, 4187), ("64x128", "one", 146, 1944, 8640), ("64x128", "pair", 155, 1984, 4279),
                  ("48x128", "three", 129, 2000, 1413), ("48x128", "pair", 130, 1968, 1456), ("80x512 64x256", "three", 600, 904, 7458), ("80x512 64x256", "pair", 1346, 920, 5223), ("112x512", "one", 1963, 904, 5952)]}


@pytest.mark.parametrize("kind, tiles, form, M, Kd, N", [(k, *t) for k, all_tiles in TILES.items() for t in all_tiles])
def test_every_tile(kind, tiles, form, M, Kd, N):
    from poptransformer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn((M, Kd), generator=g, device="cuda").half() * 0.1
    ws, dense = zip(*[weight(kind, N, Kd, g) for _ in range({"pair": 2, "three": 3}.get(form, 1))])
    outs = [torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda") for _ in range(3 if form == "three" else 1)]
    K.linear(x, list(ws), outs * 2 if form == "pair" else outs, swiglu=form == "pair")
    assert (K.linear_kernel(), K.linear_tiles(), K.linear_slices()) == ("gemm_panel_kernel", tiles, 1)
    xd, refs = x.double(), []
    for p in dense:
        ref = xd @ p.T
        refs.append((ref, 2.0 ** -11 * ref.abs() + (Kd + 2) * 2.0 ** -24 * (xd.abs() @ p.abs().T) + 2.0 ** -24))       # one rounding to fp16, sums of fp32
    if form == "pair":
        (gate, dg), (up, du) = refs
        y, swish = up.half().double(), torch.nn.functional.silu(gate)
        # fp16 up times fp16 swish of the fp16 gate: swish's slope is at most 1.1; three roundings
        bound = du * swish.abs() + (1.1 * dg + 2.0 ** -11 * (swish.abs() + 2.0 ** -14)) * (y.abs() + du) + 2.0 ** -10 * (y * swish).abs() + 2.0 ** -23
        assert ((outs[0].double() - up * swish).abs() <= bound + 2.0 ** -11 * up.abs() * swish.abs()).all()
    else:
        for out, (ref, bound) in zip(outs, refs):
            assert ((out.double() - ref).abs() <= bound).all()


# rows, features, channels; tile and slices of a product with scratch, and of one with a norm behind it whose sums may be taken in any order
@pytest.mark.parametrize("kind, M, Kd, N, alone, normed", [
    ("int4", 266, 7272, 7000, ("80x512", 4), ("80x512", 4)), ("int4", 144, 4624, 5656, ("80x256", 4), ("80x256", 4)), ("int4", 577, 8240, 816, ("64x128", 3), ("64x128", 3)),
    ("int4", 1000, 11008, 4096, ("128x512", 4), ("128x512", 4)), ("int4", 602, 4104, 4616, ("64x256", 1), ("80x512", 3)), ("int4", 133, 3136, 5712, ("48x128", 1), ("64x256", 3)),
    ("int4", 323, 4088, 2696, ("48x128", 1), ("80x128", 2)),
    ("F152", 133, 1432, 4112, ("80x512", 3), ("80x512", 3)), ("F152", 134, 2960, 4208, ("64x256", 3), ("64x256", 3)), ("F152", 133, 4048, 4224, ("48x128", 2), ("48x128", 2)),
    ("F152", 512, 1416, 6896, ("64x256", 1), ("112x512", 3)), ("F152", 268, 3184, 7192, ("80x128", 1), ("96x256", 2))])
def test_slices(kind, M, Kd, N, alone, normed):
    """Adding the slices is a launch more, but where a norm's launch makes room for it: more slices there, and only if the call allows other sums than the two calls'."""
    from poptransformer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn((M, Kd), generator=g, device="cuda").half() * 0.1
    (w, dense), gamma = weight(kind, N, Kd, g), torch.randn(N, generator=g, device="cuda").half()
    workspace = K.linear_workspace(M, N, "cuda")
    ref = x.double() @ dense.T
    bound = 2.0 ** -11 * ref.abs() + (Kd + 2) * 2.0 ** -24 * (x.double().abs() @ dense.abs().T) + 2.0 ** -24
    first, one = (torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda") for _ in range(2))
    K.linear(x, [w], [first], workspace=workspace)
    assert (K.linear_kernel(), K.linear_tiles(), K.linear_slices()) == ("gemm_panel_kernel", *alone)
    assert ((first.double() - ref).abs() <= bound).all()
    for any_order, plan in ((False, alone), (True, normed)):
        y, out = (torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda") for _ in range(2))
        K.linear_then_norm(x, w, y, K.RowNorm(gamma, None, 1e-5, out=out, any_order=any_order), workspace=workspace)
        assert (K.linear_tiles(), K.linear_slices()) == plan
        assert torch.equal(y, first) if plan == alone else ((y.double() - ref).abs() <= bound).all()
        K.rmsnorm(y, gamma, 1e-5, one)
        assert torch.equal(out, one)

"""Products of 33 rows and more by INT4 and F152 weights (gemm_panel_kernel) against float64: every tile of 48 to 128 rows with one, two and four parts of K,
slices of workgroups, and tiles of two kinds in one product; channels of any number."""
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


# features, channels, form; rows: one past 128, tiles that rows fill and that they do not, one round and several
SHAPES = {"int4": [(4096, 6144, "one"), (2056, 4096, "scratch"), (11008, 1024, "scratch"), (1032, 5632, "pair"), (520, 2048, "three"), (4104, 11008, "pair"), (8192, 6144, "one"), (4096, 1000, "one"), (1032, 50, "three"), (2048, 1303, "scratch"), (4104, 1297, "pair"), (2048, 2088, "three")],
          "F152": [(4096, 2048, "one"), (2056, 4096, "pair"), (8200, 1024, "scratch"), (1032, 1111, "pair")]}


@pytest.mark.parametrize("M", [33, 65, 128, 129, 145, 200, 333, 470, 640, 900, 1201])
@pytest.mark.parametrize("kind, Kd, N, form", [(k, *s) for k, shapes in SHAPES.items() for s in shapes])
def test_every_tile(kind, Kd, N, form, M):
    from poptransformer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn((M, Kd), generator=g, device="cuda").half() * 0.1
    ws, dense = zip(*[weight(kind, N, Kd, g) for _ in range({"pair": 2, "three": 3}.get(form, 1))])
    outs = [torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda") for _ in range(3 if form == "three" else 1)]
    K.linear(x, list(ws), outs * 2 if form == "pair" else outs, swiglu=form == "pair", workspace=K.linear_workspace(M, N, "cuda") if form == "scratch" else None)
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

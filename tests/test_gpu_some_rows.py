"""Products of 5 rows and more (gemm_own_kernel) at the edges of its tiles and of its row blocks, against float64."""
import pytest
import torch
from tests.test_gpu_many_rows import close, f8_weight, operands

pytestmark = pytest.mark.gpu

# rows at the ends of a row group; features one past, short of and on a tile of 128, with 1, 2 and an odd number of tiles for a wave and
# with waves that have none; channels short of a block, of four and of a workgroup's blocks, and odd ones
SHAPES = [(5, 8200, 250), (8, 5128, 40), (7, 13696, 72), (9, 2056, 40), (10, 3080, 264), (12, 4104, 24), (16, 5640, 1000), (16, 4096, 4112), (32, 1032, 20488), (17, 8, 16), (31, 1000, 250), (32, 1160, 264), (33, 136, 1000), (48, 2048, 272), (47, 3080, 11),
          (49, 520, 4100), (64, 4096, 2064), (63, 2176, 8200), (64, 24, 20),
          # row blocks of 48 and 64 rows, the last one with one row and full; groups of channels that are no multiple of eight
          (65, 1160, 264), (128, 4096, 4112), (129, 136, 1000), (205, 768, 2304), (256, 2056, 520), (1024, 768, 768)]


def weight_of(kind, w):
    """(weight, its numbers)"""
    from poptransformer_amd import kernels as K
    if kind == "f16":
        return K.F16Weight(w.half()), w.half().double()
    if kind == "f8":
        return f8_weight(w)
    if kind == "f152":
        scale = torch.tensor([-1], dtype=torch.int32, device="cuda")
        codes = K.half_to_fp8(w.half(), scale, "F152")
        return K.F8Weight(codes, scale, "F152"), K.fp8_to_half(codes, scale, "F152").double()
    g = torch.Generator(device="cuda").manual_seed(w.shape[0])
    packed = torch.randint(-128, 128, (w.shape[0], w.shape[1] // 2), generator=g, device="cuda", dtype=torch.int8)
    scale = (torch.rand(w.shape[0], generator=g, device="cuda") * 0.01 + 0.002).half()
    return K.W4Weight(packed, scale), K.int4_to_half(packed, scale).double().T.contiguous()


@pytest.mark.parametrize("kind", ["int4", "f16", "f8", "f152"])
@pytest.mark.parametrize("M, Kd, N", SHAPES)
@pytest.mark.parametrize("slices", [False, True])
def test_half_results(kind, M, Kd, N, slices):
    from poptransformer_amd import kernels as K
    x, w = operands(M, Kd, N, 3)
    x = x.half()
    tw, plain = weight_of(kind, w)
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    K.linear(x, [tw], [out], workspace=K.linear_workspace(M, N, "cuda") if slices else None)
    close(out, x.double() @ plain.T, x.double().abs() @ plain.abs().T, Kd, 11)


@pytest.mark.parametrize("M, N, offset", [(20, 264, 0), (33, 250, 0), (64, 264, 1), (150, 250, 1)])
def test_residual_in_place_and_results_off_their_alignment(M, N, offset):
    from poptransformer_amd import kernels as K
    Kd = 1160
    x, w = operands(M, Kd, N, 5)
    x = x.half()
    tw, plain = weight_of("int4", w)
    store = torch.randn(M * N + 1, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda").half()
    out = store[offset:offset + M * N].view(M, N)
    before = out.clone()
    K.linear(x, [tw], [out], residual=out)
    ref, mag = x.double() @ plain.T, x.double().abs() @ plain.abs().T
    # the sum is rounded, then its sum with the residual
    bound = 2.0 ** -11 * (ref.abs() + (ref + before.double()).abs()) * 1.001 + (Kd + 2) * 2.0 ** -24 * mag + 2.0 ** -23
    assert ((out.double() - ref - before.double()).abs() <= bound).all()


@pytest.mark.parametrize("kind", ["int4", "f16", "f8"])
@pytest.mark.parametrize("M", [12, 40, 130])
def test_several_matrices_with_inputs_and_biases_of_their_own(kind, M):
    from poptransformer_amd import kernels as K
    Kd, sizes = 2056, (40, 256, 270, 16)
    xs, tws, plains, biases, outs = [], [], [], [], []
    for i, n in enumerate(sizes):
        x, w = operands(M, Kd, n, 10 + i)
        tw, plain = weight_of(kind, w)
        xs.append(x.half()), tws.append(tw), plains.append(plain)
        biases.append(torch.randn(n, device="cuda").half())
        outs.append(torch.empty((M, n), dtype=torch.float16, device="cuda"))
    K.linear(None, tws, outs, biases=biases, xs=xs)
    for x, out, plain, b in zip(xs, outs, plains, biases):
        ref, mag = x.double() @ plain.T, x.double().abs() @ plain.abs().T
        bound = 2.0 ** -11 * (ref.abs() + (ref + b.double()).abs()) * 1.001 + (Kd + 2) * 2.0 ** -24 * mag + 2.0 ** -23
        assert ((out.double() - ref - b.double()).abs() <= bound).all()


@pytest.mark.parametrize("kind", ["int4", "f16", "f8"])
@pytest.mark.parametrize("M, Kd, N", [(6, 2056, 72), (16, 2048, 40), (24, 1032, 44), (48, 128, 100), (64, 2048, 4128), (12, 3080, 10008), (32, 3072, 11008), (100, 1032, 44), (129, 264, 520)])
def test_pair(kind, M, Kd, N):
    from poptransformer_amd import kernels as K
    x, w = operands(M, Kd, 2 * N, 7)
    # (the FP8 weights hold +-120, INT4 ones sums of up to 2048 * 5 * 0.1: gate and up stay far below 2^8, their product below 65504)
    x = (x if kind == "f16" else x * 0.02).half()
    (g, gp), (u, up) = weight_of(kind, w[:N].contiguous()), weight_of(kind, w[N:].contiguous())
    out = torch.empty((M, N), dtype=torch.float16, device="cuda")
    K.linear(x, [g, u], [out, out], swiglu=True)
    gate, upv = x.double() @ gp.T, x.double() @ up.T
    ref = torch.nn.functional.silu(gate) * upv
    # roundings of gate (whose error silu at most multiplies by 1.1), up, swish and the product, each 2^-11, and those of the sums
    mag_g, mag_u = x.double().abs() @ gp.abs().T, x.double().abs() @ up.abs().T
    dg, du = 2.0 ** -11 * gate.abs() + (Kd + 2) * 2.0 ** -24 * mag_g, 2.0 ** -11 * upv.abs() + (Kd + 2) * 2.0 ** -24 * mag_u
    bound = 1.1 * dg * (upv.abs() + du) + du * torch.nn.functional.silu(gate).abs() + 2.5 * 2.0 ** -11 * ref.abs() + 2.0 ** -20 * (1 + upv.abs())
    assert ((out.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("M, Kd, main, tail", [(12, 2056, 248, 5), (20, 1000, 512, 32), (64, 264, 64, 0), (40, 2048, 264, 3), (200, 520, 250, 3)])
@pytest.mark.parametrize("slices", [False, True])
def test_wide_results_with_tail(M, Kd, main, tail, slices):
    from poptransformer_amd import hybrid_kernels as HK
    x, w = operands(M, Kd, main + tail, 11)
    x, w = x.to(torch.bfloat16), w.to(torch.bfloat16)
    W = HK.WideWeight(w, torch.bfloat16, tail=tail)
    out = torch.full((M, main), float("nan"), device="cuda")
    t = torch.full((M * max(tail, 1),), float("nan"), device="cuda")
    HK.linear(x, W, out, M, ld=main, tail=t if tail else None, workspace=HK.linear_workspace(M, main + tail, "cuda") if slices else None)
    ref, mag = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    close(out, ref[:, :main], mag[:, :main], Kd, 24)
    if tail:
        close(t[:M * tail].view(M, tail), ref[:, main:], mag[:, main:], Kd, 24)


@pytest.mark.parametrize("kind", ["int4", "f16"])
def test_rows_past_the_last_and_features_past_the_end_are_not_read(kind):
    """NaN around the rows of X must not reach a result: the last row group's missing rows, and the features past K of the last tile."""
    from poptransformer_amd import kernels as K
    M, Kd, N = 35, 1032, 20
    store = torch.full((M + 64, Kd), float("nan"), dtype=torch.float16, device="cuda")
    x, w = operands(M, Kd, N, 17)
    store[:M] = x.half()
    tw, plain = weight_of(kind, w)
    out = torch.empty((M, N), dtype=torch.float16, device="cuda")
    K.linear(store[:M], [tw], [out])
    close(out, x.half().double() @ plain.T, x.half().double().abs() @ plain.abs().T, Kd, 11)


@pytest.mark.parametrize("kind, M, Kd, N", [("int4", 40, 2 ** 22 + 8, 40), ("f16", 130, 2 ** 22 + 8, 24), ("f16", 12, 2 ** 22, 24), ("int4", 64, 2 ** 25 + 8, 24)])
def test_rows_further_apart_than_32_bits_count(kind, M, Kd, N):
    """Rows of X of 8 and 64 MiB each (64 of the latter take 4 GiB): 65 features a row are +-1, so that the sums are whole numbers."""
    from poptransformer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(Kd)
    at = torch.cat([torch.randint(0, Kd - 1, (M, 64), generator=g, device="cuda"), torch.full((M, 1), Kd - 1, device="cuda")], dim=1)
    x = torch.zeros((M, Kd), dtype=torch.float16, device="cuda")
    x.scatter_(1, at, (torch.randint(0, 2, (M, 65), generator=g, device="cuda") * 2 - 1).half())
    if kind == "int4":
        packed = torch.randint(-128, 128, (N, Kd // 2), generator=g, device="cuda", dtype=torch.int8)
        tw, plain = K.W4Weight(packed, torch.ones(N, dtype=torch.float16, device="cuda")), K.int4_to_half(packed, torch.ones(N, dtype=torch.float16, device="cuda"))
    else:
        w = torch.randint(-8, 9, (N, Kd), generator=g, device="cuda", dtype=torch.int8).half()
        tw, plain = K.F16Weight(w), w.T
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    K.linear(x, [tw], [out])
    ref = (x.gather(1, at).float().unsqueeze(2) * plain[at.flatten()].view(M, 65, N).float())
    # (a feature drawn twice is in x once)
    once = torch.ones_like(at, dtype=torch.float32)
    sorted_at, order = at.sort(dim=1, stable=True)
    again = torch.cat([torch.zeros((M, 1), dtype=torch.bool, device="cuda"), sorted_at[:, 1:] == sorted_at[:, :-1]], dim=1)
    once.scatter_(1, order, (~again).float())
    assert torch.equal(out.float(), (ref * once.unsqueeze(2)).sum(1))


def test_more_channels_than_a_grid_holds():
    """Two launches: 8 * 65535 groups of three blocks of 16 channels, and the rest; channels at both ends of each, and every 100003rd."""
    from poptransformer_amd import kernels as K
    M, Kd, per = 33, 8, 8 * 65535 * 48
    N = per + 1000
    g = torch.Generator(device="cuda").manual_seed(7)
    x = torch.randn((M, Kd), generator=g, device="cuda").half()
    w = torch.randn((N, Kd), generator=g, device="cuda", dtype=torch.float16)
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    K.linear(x, [K.F16Weight(w)], [out])
    assert torch.isfinite(out).all()
    at = torch.tensor(sorted({n for e in (0, per, N) for n in range(e - 100, e + 100) if 0 <= n < N} | set(range(0, N, 100003))), device="cuda")
    close(out[:, at], x.double() @ w[at].double().T, x.double().abs() @ w[at].double().abs().T, Kd, 11)


@pytest.mark.parametrize("kind, M, Kd, N, pair, own", [
    # full steps of gemv_wide_kernel, and either side of them; channels past two blocks a compute unit; short K and long
    ("f8", 9, 4096, 4096, False, False), ("f8", 11, 4096, 1024, False, False), ("f8", 12, 4096, 4096, False, True), ("f8", 9, 3072, 4096, False, True),
    ("f8", 9, 5120, 4096, False, True), ("f8", 8, 4096, 4096, False, False), ("f8", 8, 5632, 2048, False, True), ("f8", 8, 5632, 5632, True, False),
    ("f8", 6, 8192, 4096, False, False), ("f8", 6, 11008, 4096, False, True), ("f8", 9, 4096, 5632, True, False), ("f8", 9, 4096, 2048, True, False), ("f8", 14, 4096, 2048, True, True), ("f8", 9, 9216, 2048, True, True), ("f8", 8, 1024, 2048, False, False),
    ("f16", 9, 4096, 4096, False, False), ("f16", 15, 4096, 2048, False, False), ("f16", 16, 4096, 4096, False, True), ("f16", 9, 2048, 2048, False, True),
    ("f16", 9, 5632, 2048, False, True), ("f16", 16, 4096, 4608, False, False), ("f16", 16, 2048, 2048, True, False), ("f16", 6, 11008, 4096, False, False), ("f16", 8, 8192, 2048, False, False), ("f16", 11, 12288, 1024, False, False), ("f16", 12, 8192, 2048, False, True),
    ("f16", 8, 11008, 4096, False, True), ("f8", 8, 8192, 4096, False, False), ("f8", 9, 8192, 4096, False, True), ("f8", 7, 5120, 2048, False, False),
    ("f8", 9, 2560, 12288, False, False), ("f8", 12, 2560, 12288, False, True), ("f16", 9, 5120, 4096, False, True), ("f16", 8, 5632, 2048, False, False),
    ("f152", 16, 4096, 4096, False, False), ("f152", 9, 2048, 4096, False, True), ("f152", 16, 2048, 12288, False, False), ("f152", 8, 2048, 2048, False, False),
    ("f152", 16, 11008, 4096, False, False),
    ("int4", 9, 4096, 4096, False, True), ("int4", 12, 4096, 5632, True, False), ("int4", 16, 4096, 5632, True, True), ("int4", 5, 2048, 5632, True, True),
    ("int4", 8, 2048, 11008, True, False), ("int4", 5, 4096, 24576, False, True), ("int4", 5, 4096, 12288, False, False), ("int4", 5, 8192, 2048, False, True),
    ("int4", 6, 8192, 5632, True, False)])
def test_which_few_rows_the_kernel_takes(kind, M, Kd, N, pair, own):
    taken = product(kind, M, Kd, N, pair)
    assert (taken == "gemm_own_kernel") == own, taken


def product(kind, M, Kd, N, pair):
    """A product, checked; the kernel that it took."""
    from poptransformer_amd import kernels as K
    x, w = operands(M, Kd, N, 3)
    x = (x * 0.02 if pair else x).half()
    tw, plain = weight_of(kind, w)
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    K.linear(x, [tw, tw] if pair else [tw], [out, out] if pair else [out], swiglu=pair)
    taken = K.linear_kernel()
    y, mag = x.double() @ plain.T, x.double().abs() @ plain.abs().T
    if not pair:
        close(out, y, mag, Kd, 11)
    else:
        # as in test_pair
        d = 2.0 ** -11 * y.abs() + (Kd + 2) * 2.0 ** -24 * mag
        silu = torch.nn.functional.silu(y)
        bound = 1.1 * d * (y.abs() + d) + d * silu.abs() + 2.5 * 2.0 ** -11 * (silu * y).abs() + 2.0 ** -20 * (1 + y.abs())
        assert ((out.double() - silu * y).abs() <= bound).all()
    return taken


@pytest.mark.parametrize("kind, M, Kd, N, pair, kernel", [
    # few feature tiles and several rounds, or next to none; either side of the lines
    ("f16", 33, 768, 5632, True, "gemv_mfma"), ("f16", 64, 768, 5608, True, "gemv_mfma"), ("int4", 63, 512, 8192, True, "gemv_mfma"), ("f8", 48, 768, 11008, True, "gemv_mfma"),
    ("f152", 64, 768, 8200, True, "gemv_mfma"), ("f16", 40, 512, 1000, True, "gemv_mfma"), ("f16", 48, 768, 2048, True, "gemm_own"), ("f16", 33, 1024, 5632, True, "gemm_tile"), ("f16", 33, 1024, 5608, True, "gemm_own"),
    ("f16", 40, 256, 40, False, "gemv_mfma"), ("int4", 64, 128, 1000, False, "gemv_mfma"), ("f8", 33, 8, 4104, False, "gemv_mfma"), ("f152", 49, 256, 250, False, "gemv_mfma"),
    ("f16", 33, 264, 1000, False, "gemm_own"), ("int4", 64, 768, 50257, False, "gemm_own"),
    # what gemm_tile_kernel cannot take
    ("f16", 20, 1024, 5608, True, "gemv_mfma"), ("f16", 32, 2048, 5608, True, "gemv_mfma"), ("f16", 32, 3072, 5608, True, "gemm_own"), ("f16", 17, 2048, 2056, True, "gemm_own"),
    ("int4", 20, 1024, 5608, True, "gemm_own"), 
    # F152 weights of up to 32 rows: one round of workgroups of one, two and three blocks (the last one's short of them), and the lines round it
    ("f152", 24, 2048, 1000, False, "gemv_wide"), ("f152", 17, 3072, 4104, False, "gemv_wide"), ("f152", 32, 4096, 1000, False, "gemv_wide"), ("f152", 31, 1928, 40, False, "gemv_wide"),
    ("f152", 20, 2056, 11000, False, "gemv_wide"), ("f152", 18, 4104, 12288, False, "gemv_wide"), ("f152", 32, 8200, 4104, False, "gemv_wide"), ("f152", 28, 8200, 1000, False, "gemv_wide"),
    ("f152", 29, 8200, 1000, False, "gemm_own"), ("f152", 24, 1408, 1000, False, "gemv_mfma"), ("f152", 24, 1416, 1000, False, "gemv_wide"), ("f152", 32, 1792, 4104, False, "gemv_mfma"), ("f152", 32, 1800, 4104, False, "gemv_wide"), ("f152", 24, 4096, 12304, False, "gemm_own"), ("f152", 33, 4096, 1000, False, "gemm_own"),
    ("f152", 20, 4096, 5608, True, "gemv_mfma"), ("f152", 31, 2048, 2056, True, "gemv_mfma"), ("f152", 32, 4096, 2056, True, "gemm_own"),
    ("f152", 64, 2048, 5632, True, "gemm_tile"), ("f152", 33, 1024, 5632, True, "gemm_tile"), ("f152", 40, 4096, 5632, True, "gemm_own"),
    # rounds of gemm_own_kernel beyond 64 rows
    ("int4", 65, 768, 11008, True, "gemm_rows"), ("int4", 128, 1024, 32000, False, "gemm_rows"), ("int4", 128, 2048, 5632, True, "gemm_own"),
    ("f16", 65, 8192, 8192, False, "gemm_rows"), ("f16", 65, 6144, 8192, False, "gemm_own"), ("f16", 128, 8192, 4096, False, "gemm_own"), ("f8", 100, 8192, 8192, False, "gemm_own"),
    ("int4", 65, 256, 11008, False, "gemm_own"),
    ("int4", 1000, 512, 4096, False, "gemm_panel"), ("int4", 700, 512, 4096, False, "gemm_own"), ("int4", 768, 1024, 6144, False, "gemm_panel")])
def test_which_kernel_more_rows_take(kind, M, Kd, N, pair, kernel):
    assert product(kind, M, Kd, N, pair) == kernel + "_kernel"


@pytest.mark.parametrize("M, Kd, N, pair, kernel", [(33, 256, 250, False, "gemv_mfma"), (64, 72, 1000, False, "gemv_mfma"), (40, 768, 5632, True, "gemv_mfma"),
                                                    (24, 520, 5632, True, "gemv_mfma"), (33, 520, 250, False, "gemm_own"), (65, 256, 11008, False, "gemm_rows"),
                                                    (65, 384, 11008, False, "gemm_own")])
def test_which_kernel_more_rows_of_bf16_take(M, Kd, N, pair, kernel):
    from poptransformer_amd import hybrid_kernels as HK
    x, w = operands(M, Kd, N, 11)
    x, w = (x * 0.1).to(torch.bfloat16), w.to(torch.bfloat16)
    W = HK.WideWeight(w, torch.bfloat16)
    out = torch.full((M, HK.pad8(N)), float("nan"), dtype=torch.float32, device="cuda")
    HK.linear(x, W, out, M, ld=HK.pad8(N), **(dict(up=W, pair=1) if pair else {}))
    assert HK.linear_kernel() == kernel + "_kernel"
    y, mag = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    if not pair:
        return close(out[:, :N], y, mag, Kd, 24)
    d = (Kd + 2) * 2.0 ** -24 * mag
    silu = torch.nn.functional.silu(y)
    # the sums' errors (silu multiplies the gate's by 1.1 at most), the exponential and the quotient in fp32
    bound = 1.1 * d * (y.abs() + d) + d * silu.abs() + 2.0 ** -20 * (silu * y).abs() + 2.0 ** -24
    assert ((out[:, :N].double() - silu * y).abs() <= bound).all()


@pytest.mark.parametrize("M, Kd", [(17, 2056), (32, 4104), (27, 1928)])
def test_f152_weights_over_one_input(M, Kd):
    """gemv_wide_kernel with two groups of rows: blocks of several matrices (the last workgroup's beyond them) with biases, NaN behind the last
    row; with inputs of their own and with slices of K other kernels."""
    from poptransformer_amd import kernels as K
    sizes = (40, 4096, 270, 16)
    store = torch.full((M + 32, Kd), float("nan"), dtype=torch.float16, device="cuda")
    tws, plains, biases = [], [], []
    for i, n in enumerate(sizes):
        x, w = operands(M, Kd, n, 50 + i)
        if i == 0:
            store[:M] = x.half()
        tw, plain = weight_of("f152", w)
        tws.append(tw), plains.append(plain), biases.append(torch.randn(n, device="cuda").half())
    x = store[:M]
    for xs in (None, [x] * 4):
        outs = [torch.full((M, n), float("nan"), dtype=torch.float16, device="cuda") for n in sizes]
        K.linear(None if xs else x, tws, outs, biases=biases, **(dict(xs=xs) if xs else {}))
        assert (K.linear_kernel() == "gemv_wide_kernel") == (xs is None)
        for out, plain, b in zip(outs, plains, biases):
            ref, mag = x.double() @ plain.T, x.double().abs() @ plain.abs().T
            # the sum is rounded, then its sum with the bias
            bound = 2.0 ** -11 * (ref.abs() + (ref + b.double()).abs()) * 1.001 + (Kd + 2) * 2.0 ** -24 * mag + 2.0 ** -23
            assert ((out.double() - ref - b.double()).abs() <= bound).all()
    long, w = operands(M, 11008, 1000, 60)
    tw, plain = weight_of("f152", w)
    out = torch.full((M, 1000), float("nan"), dtype=torch.float16, device="cuda")
    K.linear(long.half(), [tw], [out], workspace=K.linear_workspace(M, 1000, "cuda"))
    assert K.linear_kernel() == "gemm_own_kernel"
    close(out, long.half().double() @ plain.T, long.half().double().abs() @ plain.abs().T, 11008, 11)

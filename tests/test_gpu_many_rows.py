"""Products of more than 128 rows by 16-bit and FP8 weights, against float64.  Launches of one or few rounds go to gemm_own_kernel: the
sizes that are meant for gemm_block_kernel and gemm_rows_kernel, at the edges of their tiles, assert that they reach them (BLOCK and below)."""
import math
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [  # rows, features, channels: one past and one short of a tile of 128 / 256 rows, 64 features, 16 / 256 channels
    (129, 8, 16), (255, 72, 250), (256, 64, 256), (257, 136, 264), (384, 200, 520), (1000, 1000, 48), (513, 4096, 272),
    # more workgroups than gemm_own_kernel takes
    (129, 2056, 8200), (255, 4104, 4100), (513, 2056, 2056), (1000, 1032, 1040)]

# gemm_block_kernel: remainders of its stages of 32 and 64 features (fewer of them than it has stages, one, and past the last whole one), rows
# one past and short of 128 and 256, channels short of a block, of eight and of its groups of 256
BLOCK = [(1000, 8, 2056), (999, 24, 2050), (1000, 32, 2056), (1000, 56, 2047), (1000, 64, 2056), (897, 72, 2304), (1000, 88, 2300), (896, 96, 2560), (1000, 120, 2056),
         (129, 136, 8200), (255, 152, 8200), (256, 160, 8192), (257, 184, 8200), (383, 192, 8200), (385, 200, 8195), (1025, 520, 2056), (4096, 40, 1000)]


def close(got, ref, magnitude, K, bits):
    """One rounding of the result to `bits`, fp32 sums of K products whose magnitudes add up to `magnitude`, one subnormal step."""
    bound = 2.0 ** -bits * ref.abs() + (K + 2) * 2.0 ** -24 * magnitude + 2.0 ** -24
    worst = ((got.double() - ref).abs() / bound).max().item()
    assert worst <= 1.0, worst


def operands(M, K, N, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn((M, K), generator=g, device="cuda"), torch.randn((N, K), generator=g, device="cuda") * 0.05)


def f8_weight(w, codes_at=()):
    """F143 bytes of w with the codes at the ends of the format at some places; (weight, its numbers)."""
    from poptransformer_amd import kernels as K
    scale = torch.tensor([-1], dtype=torch.int32, device="cuda")
    codes = K.half_to_fp8(w.half(), scale)
    flat = codes.view(-1)
    for i, c in enumerate((0x7F, 0xFF, 0x01, 0x81, 0x08)):
        flat[i * 7 % flat.numel()] = c
    return K.F8Weight(codes, scale), K.fp8_to_half(codes, scale).double()


def weight_of(kind, w):
    from poptransformer_amd import kernels as K
    if kind == "f16":
        return K.F16Weight(w.half()), w.half().double()
    return f8_weight(w)


@pytest.mark.parametrize("kind", ["f16", "f8"])
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


@pytest.mark.parametrize("kind", ["f16", "f8"])
def test_several_matrices_of_any_width_with_biases(kind):
    from poptransformer_amd import kernels as K
    M, Kd, sizes = 300, 200, (40, 256, 270, 16)
    x, _ = operands(M, Kd, 1, 5)
    x = x.half()
    tws, plains, biases, outs = [], [], [], []
    for i, n in enumerate(sizes):
        tw, plain = weight_of(kind, operands(1, Kd, n, 10 + i)[1])
        tws.append(tw), plains.append(plain)
        biases.append(torch.randn(n, device="cuda").half())
        outs.append(torch.empty((M, n), dtype=torch.float16, device="cuda"))
    K.linear(x, tws, outs, biases=biases)
    for out, plain, b in zip(outs, plains, biases):
        ref = x.double() @ plain.T
        got, mag = out.double(), x.double().abs() @ plain.abs().T
        # the sum is rounded, then its sum with the bias
        bound = 2.0 ** -11 * (ref.abs() + (ref + b.double()).abs()) * 1.001 + (Kd + 2) * 2.0 ** -24 * mag + 2.0 ** -23
        assert ((got - ref - b.double()).abs() <= bound).all()


def test_inputs_of_their_own():
    from poptransformer_amd import kernels as K
    M, Kd = 200, 136
    xs = [operands(M, Kd, 1, 20 + i)[0].half() for i in range(2)]
    ws = [operands(1, Kd, n, 30 + n)[1] for n in (48, 300)]
    outs = [torch.empty((M, w.shape[0]), dtype=torch.float16, device="cuda") for w in ws]
    K.linear(None, [K.F16Weight(w.half()) for w in ws], outs, xs=xs)
    for x, w, out in zip(xs, ws, outs):
        close(out, x.double() @ w.half().double().T, x.double().abs() @ w.half().double().abs().T, Kd, 11)


@pytest.mark.parametrize("kind", ["f16", "f8"])
@pytest.mark.parametrize("M, Kd, N", [(129, 72, 40), (256, 128, 128), (515, 1032, 136), (2048, 256, 5632), (135, 2056, 4104)])
def test_pair(kind, M, Kd, N):
    from poptransformer_amd import kernels as K
    x, w = operands(M, Kd, 2 * N, 7)
    # (channel 0 of both FP8 weights holds +-120 twice: |gate|, |up| <= 4 * 120 * 5 * 0.02 = 48, the product far below 65504; with x ten
    # times that and more it would pass it)
    x = (x * 0.02 if kind == "f8" else x).half()
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


@pytest.mark.parametrize("M, Kd, main, tail", [(129, 72, 248, 5), (257, 1000, 512, 32), (1100, 264, 64, 0), (300, 2048, 264, 0), (257, 2056, 4088, 5)])
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


@pytest.mark.parametrize("M", [129, 1500])
def test_wide_group_and_sixteen_bit_results(M):
    from poptransformer_amd import hybrid_kernels as HK
    Kd = 520
    x = operands(M, Kd, 1, 13)[0].to(torch.bfloat16)
    ws = [operands(1, Kd, n, 40 + n)[1].to(torch.bfloat16) for n in (200, 24, 1024)]
    for w in ws:
        W = HK.WideWeight(w, torch.bfloat16)
        n = W.n_main
        out = torch.empty((M, HK.pad8(n)), dtype=torch.bfloat16, device="cuda")
        HK.linear(x, W, out, M)
        close(out[:, :n], x.double() @ w.double().T, x.double().abs() @ w.double().abs().T, Kd, 8)


def test_rows_past_the_last_and_features_past_the_end_are_not_read():
    """NaN around the rows of X must not reach a result: the last tile's missing rows, and the pieces past K of the last stage."""
    from poptransformer_amd import kernels as K
    M, Kd, N = 130, 24, 20
    store = torch.full((M + 300, Kd), float("nan"), dtype=torch.float16, device="cuda")
    x, w = operands(M, Kd, N, 17)
    store[:M] = x.half()
    out = torch.empty((M, N), dtype=torch.float16, device="cuda")
    K.linear(store[:M], [K.F16Weight(w.half())], [out])
    close(out, x.half().double() @ w.half().double().T, x.half().double().abs() @ w.half().double().abs().T, Kd, 11)


@pytest.mark.parametrize("slices", [False, True])
@pytest.mark.parametrize("exponent", [-140, -30, 120, 121, 127])
def test_fp8_exponents_at_the_ends_of_their_range(exponent, slices):
    """Sums of zero are zeros at every exponent whose power of two is finite; the others overflow fp16, or vanish."""
    from poptransformer_amd import kernels as K
    M, Kd, N = 1000, 1032, 2056
    x, w = operands(M, Kd, N, 19)
    x = x.half()
    x[3] = 0
    codes = K.half_to_fp8(w.half(), torch.tensor([-3], dtype=torch.int32, device="cuda"))
    codes[5] = 0
    plain = K.fp8_to_half(codes, torch.tensor([0], dtype=torch.int32, device="cuda")).double()
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    K.linear(x, [K.F8Weight(codes, torch.tensor([exponent], dtype=torch.int32, device="cuda"))], [out],
             workspace=K.linear_workspace(M, N, "cuda") if slices else None)
    s, mag = x.double() @ plain.T, x.double().abs() @ plain.abs().T
    assert (out[3] == 0).all() and (out[:, 5] == 0).all()
    sure = s.abs() > (Kd + 2) * 2.0 ** -24 * mag * 2          # the others' signs and sizes are the rounding's
    if exponent > 0:
        assert torch.equal(out[sure], (s[sure].sign() * math.inf).half())
    else:
        close(out, s * 2.0 ** exponent, mag * 2.0 ** exponent, Kd, 11)


@pytest.mark.parametrize("kind", ["f16", "f8"])
@pytest.mark.parametrize("M, Kd, N", BLOCK)
@pytest.mark.parametrize("slices", [False, True])
def test_tiles_of_both_operands_through_lds(kind, M, Kd, N, slices):
    from poptransformer_amd import kernels as K
    x, w = operands(M, Kd, N, 3)
    x = x.half()
    tw, plain = weight_of(kind, w)
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    K.linear(x, [tw], [out], workspace=K.linear_workspace(M, N, "cuda") if slices else None)
    assert K.linear_kernel() == "gemm_block_kernel"
    close(out, x.double() @ plain.T, x.double().abs() @ plain.abs().T, Kd, 11)


def test_slices_of_k_of_tiles_through_lds():
    """More slices than steps would have work for, and slices whose last one is short: the fp32 parts are added and the epilogue applied."""
    from poptransformer_amd import kernels as K
    for kind, M, Kd, N in (("f16", 1000, 4104, 1032), ("f8", 1000, 6152, 1500), ("f16", 513, 2056, 2056), ("f8", 900, 13704, 1301)):
        x, w = operands(M, Kd, N, 23)
        x = x.half()
        tw, plain = weight_of(kind, w)
        workspace = K.linear_workspace(M, N, "cuda")
        workspace.fill_(0xFF)
        bias, res = torch.randn(N, device="cuda").half(), torch.randn((M, N), device="cuda").half()
        out = res.clone()
        K.linear(x, [tw], [out], bias=bias, residual=out, workspace=workspace)
        assert K.linear_kernel() == "gemm_block_kernel"
        assert not torch.equal(workspace, torch.full_like(workspace, 0xFF))
        ref, mag = x.double() @ plain.T, x.double().abs() @ plain.abs().T
        # three roundings: the sum, with the bias, with the residual
        bound = 2.0 ** -11 * 1.001 * (ref.abs() + (ref + bias.double()).abs() + (ref + bias.double() + res.double()).abs()) + (Kd + 2) * 2.0 ** -24 * mag * 1.01 + 2.0 ** -22
        assert ((out.double() - ref - bias.double() - res.double()).abs() <= bound).all()


@pytest.mark.parametrize("kind", ["f16", "f8"])
@pytest.mark.parametrize("own_inputs", [False, True])
@pytest.mark.parametrize("M, Kd", [(1000, 200), (300, 24)])
def test_several_matrices_through_lds(kind, own_inputs, M, Kd):
    from poptransformer_amd import kernels as K
    sizes = (40, 256, 270, 8200)
    xs, tws, plains, biases, outs = [], [], [], [], []
    for i, n in enumerate(sizes):
        x, w = operands(M, Kd, n, 10 + i)
        tw, plain = weight_of(kind, w)
        xs.append(x.half()), tws.append(tw), plains.append(plain)
        biases.append(torch.randn(n, device="cuda").half())
        outs.append(torch.empty((M, n), dtype=torch.float16, device="cuda"))
    if own_inputs:
        K.linear(None, tws, outs, biases=biases, xs=xs)
    else:
        xs = xs[:1] * len(sizes)
        K.linear(xs[0], tws, outs, biases=biases)
    assert K.linear_kernel() == "gemm_block_kernel"
    for x, out, plain, b in zip(xs, outs, plains, biases):
        ref, mag = x.double() @ plain.T, x.double().abs() @ plain.abs().T
        # the sum is rounded, then its sum with the bias
        bound = 2.0 ** -11 * (ref.abs() + (ref + b.double()).abs()) * 1.001 + (Kd + 2) * 2.0 ** -24 * mag + 2.0 ** -23
        assert ((out.double() - ref - b.double()).abs() <= bound).all()


@pytest.mark.parametrize("kind", ["f16", "f8"])
@pytest.mark.parametrize("M, Kd", [(1000, 24), (999, 104), (259, 1032)])
def test_tiles_through_lds_read_nothing_past_the_rows_and_features(kind, M, Kd):
    """NaN around the rows of X: the rows that the last tile misses, and (the next row's) what lies behind a row's last feature."""
    from poptransformer_amd import kernels as K
    N = 8200
    store = torch.full((M + 300, Kd), float("nan"), dtype=torch.float16, device="cuda")
    x, w = operands(M, Kd, N, 17)
    x[::2] = x[::2].abs()
    store[:M] = x.half()
    store[M // 2] = float("nan")
    tw, plain = weight_of(kind, w)
    out = torch.empty((M, N), dtype=torch.float16, device="cuda")
    K.linear(store[:M], [tw], [out])
    assert K.linear_kernel() == "gemm_block_kernel"
    assert torch.isnan(out[M // 2]).all()
    rows = torch.arange(M, device="cuda") != M // 2
    close(out[rows], x[rows].half().double() @ plain.T, x[rows].half().double().abs() @ plain.abs().T, Kd, 11)


@pytest.mark.parametrize("kind, M, Kd, N, kernel", [
    ("f16", 129, 2048, 5632, "block"), ("f16", 160, 2048, 5632, "block"), ("f16", 200, 2056, 5632, "rows"), ("f16", 256, 2048, 2048, "rows"), ("f16", 255, 2120, 5632, "rows"),
    ("f16", 320, 2048, 3072, "rows"), ("f16", 400, 2048, 4096, "block"), ("f16", 512, 2048, 4096, "rows"), ("f16", 512, 2048, 4160, "block"), ("f16", 512, 520, 4100, "block"),
    ("f16", 1000, 2048, 2048, "block"), ("f8", 256, 2048, 5632, "block"),
    ("f8", 515, 1032, 4104, "block"), ("f8", 130, 72, 8200, "block"), ("f16", 2048, 24, 1000, "block")])
def test_which_kernel_pairs_take(kind, M, Kd, N, kernel):
    from poptransformer_amd import kernels as K
    x, w = operands(M, Kd, 2 * N, 7)
    x = (x * 0.02 if kind == "f8" else x).half()              # (as in test_pair)
    (g, gp), (u, up) = weight_of(kind, w[:N].contiguous()), weight_of(kind, w[N:].contiguous())
    out = torch.empty((M, N), dtype=torch.float16, device="cuda")
    K.linear(x, [g, u], [out, out], swiglu=True)
    assert K.linear_kernel() == f"gemm_{kernel}_kernel"
    gate, upv = x.double() @ gp.T, x.double() @ up.T
    ref = torch.nn.functional.silu(gate) * upv
    mag_g, mag_u = x.double().abs() @ gp.abs().T, x.double().abs() @ up.abs().T
    dg, du = 2.0 ** -11 * gate.abs() + (Kd + 2) * 2.0 ** -24 * mag_g, 2.0 ** -11 * upv.abs() + (Kd + 2) * 2.0 ** -24 * mag_u
    bound = 1.1 * dg * (upv.abs() + du) + du * torch.nn.functional.silu(gate).abs() + 2.5 * 2.0 ** -11 * ref.abs() + 2.0 ** -20 * (1 + upv.abs())
    assert ((out.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("M, Kd, main, tail, kernel", [
    (129, 72, 16005, 5, "block"), (257, 1000, 10990, 18, "block"), (1100, 264, 3000, 0, "block"), (520, 2048, 8200, 0, "block"), (400, 2056, 6144, 0, "block"), (1000, 40, 3200, 3, "block"),
    # short K, and one round of workgroups with whole blocks of rows
    (512, 512, 4096, 0, "rows"), (129, 1024, 6016, 128, "rows"), (512, 2048, 6140, 4, "rows"), (1000, 1000, 4096, 0, "block"), (768, 1032, 1024, 0, "block")])
@pytest.mark.parametrize("slices", [False, True])
def test_which_kernel_wide_products_take(M, Kd, main, tail, kernel, slices):
    from poptransformer_amd import hybrid_kernels as HK
    x, w = operands(M, Kd, main + tail, 11)
    x, w = x.to(torch.bfloat16), w.to(torch.bfloat16)
    W = HK.WideWeight(w, torch.bfloat16, tail=tail)
    out = torch.full((M, main), float("nan"), device="cuda")
    t = torch.full((M * max(tail, 1),), float("nan"), device="cuda")
    HK.linear(x, W, out, M, ld=main, tail=t if tail else None, workspace=HK.linear_workspace(M, W.N, "cuda") if slices else None)
    assert HK.linear_kernel() == f"gemm_{kernel}_kernel"
    ref, mag = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    close(out, ref[:, :main], mag[:, :main], Kd, 24)
    if tail:
        close(t[:M * tail].view(M, tail), ref[:, main:], mag[:, main:], Kd, 24)


@pytest.mark.parametrize("kind, M, Kd, N, kernel", [
    # K of 8192 and more, of 3072, of 2048; bf16 K past 2048 and up to it; either side of the lines
    ("f16", 200, 8192, 4096, "rows"), ("f16", 196, 8200, 4096, "block"), ("f16", 742, 6152, 2048, "rows"), ("f16", 1000, 8192, 2048, "rows"), ("f16", 1000, 4096, 4096, "block"), ("f16", 250, 3080, 4096, "rows"),
    ("f16", 320, 4096, 4096, "block"), ("f16", 250, 2056, 4096, "rows"), ("f16", 500, 2048, 4096, "block"), ("f16", 256, 1920, 12288, "block"), ("f8", 256, 8192, 12288, "block"),
    ("bf16", 192, 2056, 12288, "rows"), ("bf16", 191, 2056, 12288, "block"), ("bf16", 1000, 4096, 4096, "rows"), ("bf16", 160, 2048, 6144, "rows"), ("bf16", 129, 2048, 6144, "block"),
    ("bf16", 384, 1544, 2048, "block"), ("bf16", 250, 11008, 4096, "rows")])
def test_which_kernel_weights_take_whose_k_is_not_split(kind, M, Kd, N, kernel):
    x, w = operands(M, Kd, N, 41)
    if kind == "bf16":
        from poptransformer_amd import hybrid_kernels as HK
        x, plain = x.to(torch.bfloat16), w.to(torch.bfloat16).double()
        out = torch.full((M, N), float("nan"), device="cuda")
        HK.linear(x, HK.WideWeight(w.to(torch.bfloat16), torch.bfloat16), out, M, ld=N)
        taken, bits = HK.linear_kernel(), 24
    else:
        from poptransformer_amd import kernels as K
        x = x.half()
        tw, plain = weight_of(kind, w)
        out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
        K.linear(x, [tw], [out])
        taken, bits = K.linear_kernel(), 11
    assert taken == f"gemm_{kernel}_kernel"
    close(out, x.double() @ plain.T, x.double().abs() @ plain.abs().T, Kd, bits)


@pytest.mark.parametrize("M, Kd, N, kernel", [(256, 1024, 4096, "rows"), (129, 512, 7168, "rows"), (160, 2048, 5632, "rows"), (129, 2048, 5632, "block"), (160, 4096, 4096, "block"), (256, 4104, 4096, "rows"), (515, 136, 4100, "block")])
def test_which_kernel_wide_pairs_take(M, Kd, N, kernel):
    from poptransformer_amd import hybrid_kernels as HK
    x, w = operands(M, Kd, 2 * N, 29)
    x, w = (x * 0.1).to(torch.bfloat16), w.to(torch.bfloat16)
    g, u = (HK.WideWeight(t.contiguous(), torch.bfloat16) for t in (w[:N], w[N:]))
    out = torch.full((M, HK.pad8(N)), float("nan"), dtype=torch.bfloat16, device="cuda")
    HK.linear(x, g, out, M, ld=HK.pad8(N), up=u, pair=1)
    assert HK.linear_kernel() == f"gemm_{kernel}_kernel"
    xd, gd, ud = x.double(), w[:N].double(), w[N:].double()
    gate, upv = xd @ gd.T, xd @ ud.T
    ref = torch.nn.functional.silu(gate) * upv
    dg, du = (Kd + 2) * 2.0 ** -24 * (xd.abs() @ gd.abs().T), (Kd + 2) * 2.0 ** -24 * (xd.abs() @ ud.abs().T)
    # the sums' errors, the exponential and the quotient in fp32, one rounding to bf16
    bound = 1.1 * dg * (upv.abs() + du) + du * torch.nn.functional.silu(gate).abs() + (2.0 ** -8 + 2.0 ** -20) * ref.abs() + 2.0 ** -24
    assert ((out[:, :N].double() - ref).abs() <= bound).all()


def int4_weight(Kd, N, seed):
    from poptransformer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(seed)
    packed = torch.randint(-128, 128, (N, Kd // 2), generator=g, device="cuda", dtype=torch.int8)
    scale = (torch.rand(N, generator=g, device="cuda") * 0.01 + 0.002).half()
    return K.W4Weight(packed, scale), K.int4_to_half(packed, scale).double().T.contiguous()


@pytest.mark.parametrize("kind, M, Kd, N, kernel", [
    # registers for the rows, up to 128 of them: more rounds of gemm_own_kernel than it takes; K in slices (16-bit, few groups of channels)
    ("int4", 100, 1032, 32000, "gemm_rows_kernel"), ("int4", 128, 520, 32000, "gemm_rows_kernel"), ("int4", 65, 4096, 50304, "gemm_rows_kernel"),
    ("f16", 100, 8200, 8192, "gemm_rows_kernel"), ("f16", 128, 13704, 7168, "gemm_rows_kernel"), ("f8", 70, 1032, 40960, "gemm_rows_kernel"), ("f152", 128, 2056, 14336, "gemm_rows_kernel"),
    # panels of 128 rows: units of 64 channels that are no multiple of a workgroup's eight, or four with K in halves, so that waves have none
    ("int4", 1000, 1032, 8384, "gemm_panel_kernel"), ("int4", 1000, 2056, 6464, "gemm_panel_kernel"), ("int4", 4096, 4096, 320, "gemm_panel_kernel"), ("int4", 3000, 8200, 448, "gemm_panel_kernel"),
    ("int4", 1025, 4104, 2112, "gemm_panel_kernel"), ("f152", 600, 2056, 4160, "gemm_panel_kernel"),
    # blocks that do not divide: 64 rows in turn, the last eight
    ("int4", 200, 1032, 32008, "gemv_"), ("f152", 136, 520, 32040, "gemv_")])
@pytest.mark.parametrize("slices", [False, True])
def test_kernels_of_many_rounds(kind, M, Kd, N, kernel, slices):
    from poptransformer_amd import kernels as K
    x, w = operands(M, Kd, 8 if kind == "int4" else N, 31)
    x = x.half()
    if kind == "int4":
        tw, plain = int4_weight(Kd, N, 33)
    elif kind == "f152":
        scale = torch.tensor([-1], dtype=torch.int32, device="cuda")
        codes = K.half_to_fp8(w.half(), scale, "F152")
        tw, plain = K.F8Weight(codes, scale, "F152"), K.fp8_to_half(codes, scale, "F152").double()
    else:
        tw, plain = weight_of(kind, w)
    workspace = K.linear_workspace(M, N, "cuda") if slices else None
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    K.linear(x, [tw], [out], workspace=workspace)
    assert K.linear_kernel().startswith(kernel), K.linear_kernel()
    ref, mag = x.double() @ plain.T, x.double().abs() @ plain.abs().T
    close(out, ref, mag, Kd, 11)
    # in place on the residual, behind a bias
    bias, res = torch.randn(N, device="cuda").half(), torch.randn((M, N), device="cuda").half()
    out = res.clone()
    K.linear(x, [tw], [out], bias=bias, residual=out, workspace=workspace)
    bound = 2.0 ** -11 * 1.001 * (ref.abs() + (ref + bias.double()).abs() + (ref + bias.double() + res.double()).abs()) + (Kd + 2) * 2.0 ** -24 * mag * 1.01 + 2.0 ** -22
    assert ((out.double() - ref - bias.double() - res.double()).abs() <= bound).all()


def test_panels_of_a_pair_and_of_several_matrices():
    """Units of pairs and of matrices that share a workgroup with idle waves; the last round of tiles in a launch of its own."""
    from poptransformer_amd import kernels as K
    for M, Kd, N in ((1000, 1032, 4192), (600, 2056, 2080)):
        x = (operands(M, Kd, 1, 35)[0] * 0.02).half()
        (g, gp), (u, up) = int4_weight(Kd, N, 36), int4_weight(Kd, N, 37)
        out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
        K.linear(x, [g, u], [out, out], swiglu=True)
        assert K.linear_kernel() == "gemm_panel_kernel"
        gate, upv = x.double() @ gp.T, x.double() @ up.T
        silu = torch.nn.functional.silu(gate)
        dg, du = (2.0 ** -11 * t.abs() + (Kd + 2) * 2.0 ** -24 * (x.double().abs() @ p.abs().T) for t, p in ((gate, gp), (upv, up)))
        # as in test_pair
        bound = 1.1 * dg * (upv.abs() + du) + du * silu.abs() + 2.5 * 2.0 ** -11 * (silu * upv).abs() + 2.0 ** -20 * (1 + upv.abs())
        assert ((out.double() - silu * upv).abs() <= bound).all()
    M, Kd, sizes = 900, 1032, (4160, 320, 4096, 192)
    x = operands(M, Kd, 1, 38)[0].half()
    ws = [int4_weight(Kd, n, 40 + i) for i, n in enumerate(sizes)]
    outs = [torch.full((M, n), float("nan"), dtype=torch.float16, device="cuda") for n in sizes]
    K.linear(x, [w for w, _ in ws], outs)
    assert K.linear_kernel() == "gemm_panel_kernel"
    for (_, p), out in zip(ws, outs):
        close(out, x.double() @ p.T, x.double().abs() @ p.abs().T, Kd, 11)


# The ends of gemm_block_kernel and gemm_panel_kernel: sizes that are stored straight from the registers (channels in eights, few kinds of ends) and
# beside each one that is not; rows one past and one short of a row group, channels short of a wave's tile.
ENDS = [(1025, 520, 2056), (1009, 520, 2052), (1039, 200, 2050), (4096, 40, 1000)]


@pytest.mark.parametrize("kind", ["f16", "f8", "int4"])
@pytest.mark.parametrize("M, Kd, N", ENDS)
@pytest.mark.parametrize("bias, residual, act", [(0, 1, 0), (1, 0, 0), (1, 1, 0), (1, 1, 1)])
def test_ends_of_half_results(kind, M, Kd, N, bias, residual, act):
    from poptransformer_amd import _lib
    from poptransformer_amd import kernels as K
    x, w = operands(M, Kd, N, 41)
    # (a channel of the FP8 weight holds +-120 and more five times: the sum stays below 5 * 240 * 5.5 * 0.02 = 132 and the square of it and a bias below 20000, where
    # with x fifty times that it passes 65504)
    x = (x * 0.02 if kind == "f8" else x).half()
    if kind == "int4":
        N = N // 8 * 8
        w = w[:N]
        scale = (w.abs().amax(1) / 7.0).half()
        q = torch.clamp(torch.round(w / scale.float()[:, None]), -8, 7).to(torch.int8)
        u = (q & 0xF).to(torch.uint8)
        tw, plain = K.W4Weight(((u[:, 0::2] << 4) | u[:, 1::2]).view(torch.int8).contiguous(), scale), (q.half() * scale[:, None]).double()
    else:
        tw, plain = weight_of(kind, w)
    b, r = torch.randn(N, device="cuda").half(), torch.randn((M, N), device="cuda").half()
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    K.linear(x, [tw], [out], bias=b if bias else None, residual=r if residual else None, act=_lib.ACT_RELU_SQUARE if act else _lib.ACT_NONE)
    ref, mag = x.double() @ plain.T, x.double().abs() @ plain.abs().T
    error = 2.0 ** -11 * ref.abs() + (Kd + 2) * 2.0 ** -24 * mag + 2.0 ** -24              # of the rounded sum, then of each step on it
    if bias:
        ref = ref + b.double()
        error = error + 2.0 ** -11 * (ref.abs() + error)
    if act:
        ref, slope = torch.relu(ref) ** 2, 2 * torch.relu(ref)
        error = error * (slope + error) + 2.0 ** -11 * (ref + error)
    if residual:
        ref = ref + r.double()
        error = error + 2.0 ** -11 * (ref.abs() + error)
    assert ((out.double() - ref).abs() <= error * 1.001 + 2.0 ** -23).all()


@pytest.mark.parametrize("M, Kd, N", ENDS)
@pytest.mark.parametrize("end", ["plain", "sigmoid", "gelu", "fp32", "added", "product", "cap", "pair", "clamped", "pair_biases"])
def test_ends_of_wide_results(M, Kd, N, end):
    from poptransformer_amd import _hybrid_lib as H
    from poptransformer_amd import hybrid_kernels as HK
    x, w = operands(M, Kd, 2 * N, 43)
    x, w, F = x.bfloat16(), w.bfloat16(), torch.nn.functional
    ld = HK.pad8(N)
    made = [HK.WideWeight(w[i * N:(i + 1) * N].float(), torch.bfloat16, main_to=ld if "pair" in end or end == "clamped" else None) for i in (0, 1)]
    g, u = (x.double() @ w[i * N:(i + 1) * N].double().T for i in (0, 1))
    b1, b2 = torch.randn(ld, device="cuda"), torch.randn(ld, device="cuda")
    f32 = end in ("fp32", "added", "product", "cap")
    out = torch.randn((M, ld), device="cuda").to(torch.float32 if f32 else torch.bfloat16)
    by, before = torch.randn((M, ld), device="cuda").bfloat16(), out.double()
    kw = {"plain": {}, "sigmoid": dict(bias=b1, act=H.ACT_SIGMOID), "gelu": dict(act=H.ACT_GELU_TANH), "fp32": dict(bias=b1), "cap": dict(cap=1.5),
          "added": dict(bias=b1, accumulate=True), "product": dict(mul=by, accumulate=True), "pair": dict(up=made[1], pair=H.PAIR_SWIGLU),
          "clamped": dict(up=made[1], pair=H.PAIR_CLAMPED, limit=1.25, slope=1.7), "pair_biases": dict(up=made[1], pair=H.PAIR_SWIGLU, bias=b1, bias2=b2)}[end]
    if N % 8 and end in ("sigmoid", "fp32", "added"):                                       # (a bias has a number for every main channel)
        kw["bias"] = b1[:N].contiguous()
    HK.linear(x, made[0], out, M, ld=ld, **kw)
    v, up, B1, B2 = g, u, b1[:N].double(), b2[:N].double()
    ref = {"plain": lambda: v, "sigmoid": lambda: torch.sigmoid(v + B1), "gelu": lambda: F.gelu(v, approximate="tanh"), "fp32": lambda: v + B1,
           "cap": lambda: 1.5 * torch.tanh(v / 1.5), "added": lambda: before[:, :N] + v + B1, "product": lambda: before[:, :N] + v * by[:, :N].double(),
           "pair": lambda: F.silu(v) * up, "pair_biases": lambda: F.silu(v + B1) * (up + B2),
           "clamped": lambda: v.clamp(max=1.25) * torch.sigmoid(1.7 * v.clamp(max=1.25)) * (up.clamp(-1.25, 1.25) + 1)}[end]()
    # sums of K products (numbers of about 0.05 sqrt(K)) in fp32, at most multiplied by the other factor; one rounding to bf16
    factor = 1 + (by[:, :N].double().abs() if end == "product" else (v.abs() + up.abs() + 4) if "pair" in end or end == "clamped" else 1)
    mag = (x.double().abs() @ w[:N].double().abs().T).amax()
    bound = (0 if f32 else 2.0 ** -8) * ref.abs() + (Kd + 8) * 2.0 ** -24 * mag * factor + 4 * 2.0 ** -24 * ref.abs() + 2.0 ** -24
    worst = ((out[:, :N].double() - ref).abs() / bound).max().item()
    assert worst <= 1.0, worst
    if ld > N and "pair" not in end and end != "clamped":
        assert torch.equal(out[:, N:].double(), before[:, N:])                              # columns past the last channel are left alone


# gemm_block_kernel's tiles, alone and behind whole rounds of 256 rows: rows one past a tile, channels short of a block and of a tile
TILES = [("one", 1537, 200, 5000, "192x256"), ("one", 385, 72, 5003, "128x128"), ("one", 641, 200, 4100, "128x128"), ("pair", 385, 2056, 1500, "128x128"), ("one", 1921, 1032, 8195, "256x256 128x128"), ("one", 1921, 2056, 12300, "256x256 192x256"),
         ("pair", 257, 200, 11000, "256x256"), ("pair", 385, 520, 1500, "128x128"), ("pair", 385, 72, 8195, "192x256"), ("pair", 129, 72, 8195, "128x256"),
         ("pair", 1537, 1032, 5000, "256x256 128x128"), ("pair", 1537, 72, 11000, "256x256 128x256"), ("pair", 1921, 2056, 6152, "256x256 192x256"),
         ("three", 1153, 200, 2051, "192x256"), ("three", 577, 136, 1030, "128x128"), ("three", 961, 72, 11000, "256x256 128x256"), ("three", 1921, 2056, 4100, "256x256 192x256")]


@pytest.mark.parametrize("kind", ["f16", "f8", "bf16"])
@pytest.mark.parametrize("form, M, Kd, N, tiles", TILES)
def test_tiles_of_other_sizes(kind, form, M, Kd, N, tiles):
    from poptransformer_amd import hybrid_kernels as HK
    from poptransformer_amd import kernels as K
    if kind == "bf16" and form == "three":
        pytest.skip("the wide entry point takes several weights of few rows only")
    x, w = operands(M, Kd, {"one": 1, "pair": 2, "three": 3}[form] * N, 51)
    parts = [w[i * N:(i + 1) * N] for i in range(w.shape[0] // N)]
    if kind == "bf16":
        x, ld = x.bfloat16(), HK.pad8(N)
        plains = [p.bfloat16().double() for p in parts]
        tws = [HK.WideWeight(p, torch.bfloat16, main_to=ld if form == "pair" else None) for p in parts]
        out = torch.full((M, ld), float("nan"), dtype=torch.bfloat16 if form == "pair" else torch.float32, device="cuda")
        if form == "pair":
            from poptransformer_amd import _hybrid_lib as H
            HK.linear(x, tws[0], out, M, ld=ld, up=tws[1], pair=H.PAIR_SWIGLU)
        else:
            HK.linear(x, tws[0], out, M, ld=ld)
        if (M, Kd, N) in ((385, 72, 5003), (385, 520, 1500)):                                              # (few tiles and short K: bf16 has another kernel for them)
            assert HK.linear_kernel() == "gemm_rows_kernel"
        else:
            assert (HK.linear_kernel(), HK.linear_tiles()) == ("gemm_block_kernel", tiles)
        outs = [out[:, :N]]
    else:
        x = (x * 0.02 if kind == "f8" and form == "pair" else x).half()                     # (as in test_pair: the product stays far below 65504)
        tws, plains = zip(*(weight_of(kind, p) for p in parts))
        outs = [torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda") for _ in range(3 if form == "three" else 1)]
        K.linear(x, list(tws), outs * 2 if form == "pair" else outs, swiglu=form == "pair")
        assert (K.linear_kernel(), K.linear_tiles()) == ("gemm_block_kernel", tiles)
    if form != "pair":
        for out, plain in zip(outs, plains):
            close(out, x.double() @ plain.T, x.double().abs() @ plain.abs().T, Kd, 24 if kind == "bf16" else 11)
        return
    gate, upv = (x.double() @ p.T for p in plains)
    silu = torch.nn.functional.silu(gate)
    unit = 0.0 if kind == "bf16" else 2.0 ** -11                                            # (fp16 results are rounded before the activation as well)
    dg, du = (unit * t.abs() + (Kd + 2) * 2.0 ** -24 * (x.double().abs() @ p.abs().T) for t, p in ((gate, plains[0]), (upv, plains[1])))
    # as in test_pair: the slope of silu is below 1.1; swish and the product are rounded
    last = 2.0 ** -8 if kind == "bf16" else 2.5 * 2.0 ** -11
    bound = 1.1 * dg * (upv.abs() + du) + du * silu.abs() + last * (silu * upv).abs() + 2.0 ** -20 * (1 + upv.abs())
    assert ((outs[0].double() - silu * upv).abs() <= bound).all()


@pytest.mark.parametrize("form, M, Kd, N", [("one", 1000, 328, 2100), ("one", 600, 13704, 2100), ("slices", 1500, 2056, 1040), ("pair", 900, 200, 1500)])
def test_blocks_of_fp8_channels_with_the_largest_codes(form, M, Kd, N):
    """A few blocks of channels that hold 0x7F or 0xFF (+-240, which the fast conversion does not know) in their first, a middle and their last tile: they are right,
    and the channels of all others are bit for bit what they are beside weights without these codes."""
    from poptransformer_amd import kernels as K
    x, w = operands(M, Kd, 2 * N, 61)
    x = (x * 0.02).half()
    scale = torch.tensor([-1], dtype=torch.int32, device="cuda")
    codes = K.half_to_fp8(w.half(), scale)
    assert not ((codes.view(torch.uint8) & 0x7F) == 0x7F).any()
    marked = codes.clone()
    flat = marked.view(torch.uint8)
    at = [(3, 0), (N // 2, Kd // 2), (N - 1, Kd - 1), (N + 40, Kd // 3)]
    for i, (n, k) in enumerate(at):
        flat[n, k] = 0x7F if i % 2 else 0xFF
    outs = []
    for c in (codes, marked):
        ws = [K.F8Weight(c[i * N:(i + 1) * N].contiguous(), scale) for i in range(2 if form == "pair" else 1)]
        out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
        K.linear(x, ws, [out] * len(ws), swiglu=form == "pair", workspace=K.linear_workspace(M, N, "cuda") if form == "slices" else None)
        assert K.linear_kernel() == "gemm_block_kernel"
        outs.append(out)
    plain = K.fp8_to_half(marked, scale).double()
    # (a wave's channels, four blocks of a matrix or two of each of a pair's, are converted one way together)
    assert torch.equal(outs[0][:, 128:N // 2 - 128], outs[1][:, 128:N // 2 - 128]) and torch.equal(outs[0][:, N // 2 + 128:N - 128], outs[1][:, N // 2 + 128:N - 128])
    xd = x.double()
    if form != "pair":
        close(outs[1], xd @ plain[:N].T, xd.abs() @ plain[:N].abs().T, Kd, 11)
        return
    gate, upv = xd @ plain[:N].T, xd @ plain[N:].T
    silu = torch.nn.functional.silu(gate)
    dg, du = (2.0 ** -11 * t.abs() + (Kd + 2) * 2.0 ** -24 * (xd.abs() @ p.abs().T) for t, p in ((gate, plain[:N]), (upv, plain[N:])))
    bound = 1.1 * dg * (upv.abs() + du) + du * silu.abs() + 2.5 * 2.0 ** -11 * (silu * upv).abs() + 2.0 ** -20 * (1 + upv.abs())      # as in test_pair
    assert ((outs[1].double() - silu * upv).abs() <= bound).all()


def test_every_gate_comes_out_as_by_the_operator():
    """Every fp16 gate but NaN through the end of a tile, bit for bit: rows that pick one feature, so that sums are the weights' own values, beside 1 from the
    other weight."""
    from poptransformer_amd import kernels as K
    gates = torch.arange(-32768, 32768, dtype=torch.int32, device="cuda").to(torch.int16).view(torch.float16)
    gates = gates[~torch.isnan(gates) & (gates.view(torch.int16) != -32768)]      # (a sum has no negative zero)
    gates = torch.cat([gates, gates.new_ones(-len(gates) % 8)])
    x = torch.zeros((136, 32), dtype=torch.float16, device="cuda")
    x[:, 5] = 1
    g, u = torch.zeros((2, len(gates), 32), dtype=torch.float16, device="cuda")
    g[:, 5], u[:, 5] = gates, 1
    out = torch.full((136, len(gates)), 7.0, dtype=torch.float16, device="cuda")
    K.linear(x, [K.F16Weight(g), K.F16Weight(u)], [out, out], swiglu=True)
    assert K.linear_kernel() == "gemm_block_kernel"
    want = K.swiglu(gates, torch.ones_like(gates))
    differ = ((out.view(torch.int16) != want.view(torch.int16)) & ~(torch.isnan(out) & torch.isnan(want))).any(0)
    assert not differ.any(), (gates[differ], out[0, differ], want[differ])


@pytest.mark.parametrize("end", ["sigmoid", "swiglu", "clamped"])
def test_activations_do_not_depend_on_how_many_rows_there_are(end):
    """The same sums, exact by rows that pick one feature, through the kernels of few and of many rows: gates of all fp32 fractions from -60 to 60."""
    from poptransformer_amd import _hybrid_lib as H
    from poptransformer_amd import hybrid_kernels as HK
    N = 262144
    x = torch.zeros((264, 64), dtype=torch.bfloat16, device="cuda")
    x[:, 9] = 1
    w = torch.zeros((2, N, 64), device="cuda")
    w[1, :, 9] = torch.linspace(-3, 3, N, device="cuda").bfloat16().float()
    made = [HK.WideWeight(t, torch.bfloat16) for t in w]
    b1, b2 = torch.linspace(-60, 60, N, device="cuda") * 1.0003, torch.linspace(-1, 1, N, device="cuda")
    kw = {"sigmoid": dict(bias=b1, act=H.ACT_SIGMOID), "swiglu": dict(up=made[1], pair=H.PAIR_SWIGLU, bias=b1, bias2=b2),
          "clamped": dict(up=made[1], pair=H.PAIR_CLAMPED, limit=7.0, slope=1.7, bias=b1, bias2=b2)}[end]
    results = {}
    for rows in (4, 16, 264):
        out = torch.full((rows, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        HK.linear(x, made[0], out, rows, ld=N, **kw)
        results[HK.linear_kernel()] = out[:1]
        assert torch.equal(out, out[:1].expand_as(out))
    assert "gemm_block_kernel" in results and len(results) > 1
    for out in results.values():
        differ = (out != results["gemm_block_kernel"]).sum().item()
        assert differ == 0, differ

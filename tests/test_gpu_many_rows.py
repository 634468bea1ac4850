"""Products of more than 128 rows by 16-bit and FP8 weights (gemm_block_kernel) at the edges of its tiles, against float64."""
import math
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [  # rows, features, channels: one past and one short of a tile of 128 / 256 rows, 64 features, 16 / 256 channels
    (129, 8, 16), (255, 72, 250), (256, 64, 256), (257, 136, 264), (384, 200, 520), (1000, 1000, 48), (513, 4096, 272),
    # more workgroups than gemm_own_kernel takes
    (129, 2056, 8200), (255, 4104, 4100), (513, 2056, 2056), (1000, 1032, 1040)]


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

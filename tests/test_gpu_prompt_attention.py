"""prompt_attention_mfma_kernel at the ends of its row groups, workgroups and steps of 64 cache rows, against float64."""
import math
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # sequences, rows, query heads, KV heads, ring, step
    (1, 16, 1, 1, 16, 0), (1, 17, 8, 8, 64, 0), (2, 63, 5, 5, 128, 0), (1, 64, 9, 3, 130, 65), (3, 65, 12, 4, 200, 63), (1, 129, 16, 2, 192, 40),
    (2, 128, 7, 7, 100, 20), (1, 300, 32, 32, 512, 1),
    # one step: of 20, 32, 33 and 64 cache rows, and one row more than that; a ring that is full before the pass
    (1, 20, 3, 3, 20, 30), (1, 32, 3, 3, 40, 0), (2, 33, 4, 2, 64, 0), (1, 17, 9, 3, 64, 47), (1, 64, 3, 3, 64, 9), (2, 16, 3, 3, 80, 49)]


@pytest.mark.parametrize("kv8", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B, rows, Hq, Hkv, ring, step", [c for c in CASES if c[1] <= c[4]])
@pytest.mark.parametrize("offset", [0, 1])
def test_against_float64(B, rows, Hq, Hkv, ring, step, D, kv8, offset):
    from poptransformer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(rows)
    randn = lambda *s: torch.randn(s, generator=g, device="cuda")
    q = randn(B, rows, Hq, D).half()
    # rows of the ring past the last valid one hold NaN (F143 has none: its largest value)
    n = min(step + rows, ring)
    if kv8:
        codes = K.half_to_fp8(randn(2 * B * Hkv * ring, D).half(), torch.tensor([0], dtype=torch.int32, device="cuda"), "F143").view(2, B, Hkv, ring, D)
        codes[:, :, :, n:] = 0x7F
        kv = K.fp8_to_half(codes.view(-1, D), torch.tensor([0], dtype=torch.int32, device="cuda"), "F143").view(codes.shape)
    else:
        kv = codes = randn(2, B, Hkv, ring, D).half()
        codes[:, :, :, n:] = float("nan")
    store = torch.full((B * rows * Hq * D + 1,), float("nan"), dtype=torch.float16, device="cuda")
    out = store[offset:offset + B * rows * Hq * D].view(B, rows, Hq, D)
    K.prompt_attention(q, codes, torch.tensor(step, dtype=torch.int32, device="cuda"), K.decode_attention_workspace(B * rows, Hq, D, ring, "cuda"), out,
                       B, rows, Hq, Hkv, D, ring, True, kv_scale=0 if kv8 else None)
    k, v = (t[:, :, :n].double().repeat_interleave(Hq // Hkv, dim=1) for t in kv)
    scale = torch.tensor(1 / math.sqrt(D), dtype=torch.float16, device="cuda")
    s = ((q.double().transpose(1, 2).contiguous().float() @ k.transpose(2, 3).contiguous().float()).half() * scale).double()
    valid = torch.clamp(torch.arange(rows, device="cuda") + step + 1, max=ring)
    seen = torch.arange(n, device="cuda")[None, :] < valid[:, None]
    p = torch.softmax(s.masked_fill(~seen, -math.inf), dim=-1)
    ref, mag = p @ v, p @ v.abs()
    # the probabilities' rounding (2^-11, below 2^-14 steps of 2^-25 on numbers whose largest is 1), the result's, fp32 sums; a score whose sum
    # rounds to the other fp16 neighbour, and then its product with the scale, moves its probability by 2 * 2^-10 of the score
    top = s.masked_fill(~seen, 0).abs().amax(-1, keepdim=True)
    bound = (2.0 ** -11 * 2 + 4 * 2.0 ** -10 * top + n * 2.0 ** -20) * mag + n * 2.0 ** -25 * v.abs().amax() + 2.0 ** -24
    got = out.double().transpose(1, 2)
    assert torch.isfinite(got).all()
    assert ((got - ref).abs() <= bound).all(), ((got - ref).abs() / bound).max().item()


def test_a_head_whose_cache_rows_take_more_than_4_gib():
    """The last 16 of 2^25 + 200 positions: four rows of the ring, one of them past the first 4 GiB, share all of the weight (scores of 40
    against 0: the others' weights, 2^25 * e^-40 of 4, lie below 2^-30), so the result is the mean of their V rows."""
    from poptransformer_amd import kernels as K
    D, rows, n = 64, 16, 2 ** 25 + 200
    assert 2 ** 25 * D * 2 >= 2 ** 32
    kv = torch.zeros((2, 1, 1, n, D), dtype=torch.float16, device="cuda")
    at = torch.tensor([5, 2 ** 24 + 3, 2 ** 25 + 7, n - 20], device="cuda")
    kv[0, 0, 0, at] = 5.0
    v = torch.randn((4, D), generator=torch.Generator(device="cuda").manual_seed(1), device="cuda").half()
    kv[1, 0, 0, at] = v
    q = torch.ones((1, rows, 1, D), dtype=torch.float16, device="cuda")
    out = torch.full((1, rows, 1, D), float("nan"), dtype=torch.float16, device="cuda")
    K.prompt_attention(q, kv, torch.tensor(n - rows, dtype=torch.int32, device="cuda"), K.decode_attention_workspace(rows, 1, D, n, "cuda"), out,
                       1, rows, 1, 1, D, n, True)
    ref = v.double().mean(0)
    # weights of exactly 1 (fp16), a sum of 4 in fp32, one rounding of the quotient; the rest of the weights
    bound = 2.0 ** -11 * ref.abs() + 2.0 ** -24 + 2.0 ** -28 * v.double().abs().amax()
    assert ((out.double().view(rows, D) - ref).abs() <= bound).all()


def test_more_heads_than_a_grid_holds():
    """Three launches (8 * 65535 heads each, the last one of 30), heads past 2^20 (whose quotients are integer divisions), grouped KV heads;
    the heads on either side of the launches' ends and of 2^20, the first and last ones of a sequence, and every 9973rd."""
    from poptransformer_amd import kernels as K
    B, Hq, Hkv, D, rows = 3, 349530, 5, 64, 16
    heads = B * Hq
    assert heads == 2 * 8 * 65535 + 30 and heads > 2 ** 20
    g = torch.Generator(device="cuda").manual_seed(3)
    q = torch.randn((B, rows, Hq, D), generator=g, device="cuda", dtype=torch.float16)
    kv = torch.randn((2, B, Hkv, rows, D), generator=g, device="cuda", dtype=torch.float16)
    out = torch.full((B, rows, Hq, D), float("nan"), dtype=torch.float16, device="cuda")
    K.prompt_attention(q, kv, torch.tensor(0, dtype=torch.int32, device="cuda"), K.decode_attention_workspace(B * rows, Hq, D, rows, "cuda"), out,
                       B, rows, Hq, Hkv, D, rows, True)
    assert torch.isfinite(out).all()
    ends = [i * 8 * 65535 for i in range(3)] + [2 ** 20, Hq, 2 * Hq, heads]
    at = torch.tensor(sorted({h for e in ends for h in range(e - 9, e + 9) if 0 <= h < heads} | set(range(0, heads, 9973))), device="cuda")
    b, h = at // Hq, at % Hq
    k, v = (t[b, h // (Hq // Hkv)].double() for t in kv)
    s = (q[b, :, h].float() @ k.transpose(1, 2).contiguous().float()).half() * torch.tensor(1 / math.sqrt(D), dtype=torch.float16, device="cuda")
    seen = torch.arange(rows, device="cuda")[None, :] <= torch.arange(rows, device="cuda")[:, None]
    p = torch.softmax(s.double().masked_fill(~seen, -math.inf), dim=-1)
    # the bound of test_against_float64
    bound = (2.0 ** -11 * 2 + 4 * 2.0 ** -10 * s.double().abs().amax(-1, keepdim=True) + rows * 2.0 ** -20) * (p @ v.abs()) + rows * 2.0 ** -25 * v.abs().amax() + 2.0 ** -24
    assert ((out[b, :, h].double() - p @ v).abs() <= bound).all()


@pytest.mark.parametrize("kv8", [False, True])
@pytest.mark.parametrize("step", [0, 64])
def test_infinities_ahead_do_not_reach_rows_32_positions_behind(kv8, step):
    """V holds an infinity (F143: its largest value) at position step + 40: rows whose waves end before the 32 cache rows that hold it are
    what they are without it."""
    from poptransformer_amd import kernels as K
    D, rows, heads, ring = 64, 64, 3, 192
    g = torch.Generator(device="cuda").manual_seed(5)
    q = torch.randn((1, rows, heads, D), generator=g, device="cuda").half()
    kv = torch.randn((2, 1, heads, ring, D), generator=g, device="cuda").half()
    bad = kv.clone()
    bad[1, :, :, step + 40] = float("inf")
    outs = []
    for t in (kv, bad):
        t = K.half_to_fp8(t.view(-1, D), torch.tensor([0], dtype=torch.int32, device="cuda"), "F143").view(kv.shape) if kv8 else t
        out = torch.full((1, rows, heads, D), float("nan"), dtype=torch.float16, device="cuda")
        K.prompt_attention(q, t, torch.tensor(step, dtype=torch.int32, device="cuda"), K.decode_attention_workspace(rows, heads, D, ring, "cuda"),
                           out, 1, rows, heads, heads, D, ring, True, kv_scale=0 if kv8 else None)
        outs.append(out)
    assert torch.isfinite(outs[1][:, :32]).all()
    assert torch.equal(outs[0][:, :32], outs[1][:, :32])

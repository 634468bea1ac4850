"""F143 weights that hold none of the codes 0x7F, 0xFF and 0x80 go to kernels of their own (PTA_W_F143_PLAIN), whose conversion is the hardware's: the same numbers, and the
same results as by the kernels for all codes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def scale():
    return torch.tensor([-1], dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("rows", [1, 8, 40, 300])
def test_every_code(rows):
    from poptransformer_amd import kernels as K
    codes = torch.tensor([c for c in range(256) if c not in (0x7F, 0xFF, 0x80)], dtype=torch.uint8, device="cuda")
    w8 = torch.zeros((len(codes), 32), dtype=torch.uint8, device="cuda")
    w8[:, 7] = codes
    w = K.F8Weight(w8, scale())
    assert w.plain
    x = torch.zeros((rows, 32), dtype=torch.float16, device="cuda")
    x[:, 7] = 1
    out = torch.full((rows, len(codes)), float("nan"), dtype=torch.float16, device="cuda")
    K.linear(x, [w], [out])
    assert torch.equal(out, K.fp8_to_half(codes, scale()).expand_as(out))


@pytest.mark.parametrize("kind, Kd, N", [("one", 4096, 4100), ("one", 200, 136), ("one", 13704, 520), ("slices", 2048, 1024), ("pair", 4096, 4096), ("three", 1032, 2050)])
@pytest.mark.parametrize("rows", [1, 4, 5, 8, 16, 17, 33, 64, 65, 128, 129, 500])
def test_like_the_kernels_for_all_codes(kind, Kd, N, rows):
    from poptransformer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(rows)
    n = {"pair": 2, "three": 3}.get(kind, 1)
    x = (torch.randn((rows, Kd), generator=g, device="cuda") * 0.2).half()
    ws = [K.F8Weight(K.half_to_fp8((torch.randn((N, Kd), generator=g, device="cuda") * 0.02).half(), scale()), scale()) for _ in range(n)]
    results = []
    for plain in (True, False):
        for w in ws:
            assert w.plain or plain is False
            w.plain = plain
        outs = [torch.full((rows, N), float("nan"), dtype=torch.float16, device="cuda") for _ in range(3 if kind == "three" else 1)]
        K.linear(x, ws, outs * 2 if kind == "pair" else outs, swiglu=kind == "pair", workspace=K.linear_workspace(rows, N, "cuda") if kind == "slices" else None)
        results.append((K.linear_kernel(), outs))
    assert results[0][0] == results[1][0]
    for a, b in zip(results[0][1], results[1][1]):
        assert torch.equal(a, b)


@pytest.mark.parametrize("rows", [2, 8, 64, 260])
def test_codes_beyond_the_conversion(rows):
    """Such a weight is not called plain, also beside one that is."""
    from poptransformer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(5)
    Kd, N = 1024, 512
    x = (torch.randn((rows, Kd), generator=g, device="cuda") * 0.05).half()
    codes = [K.half_to_fp8((torch.randn((N, Kd), generator=g, device="cuda") * 0.02).half(), scale()) for _ in range(2)]
    codes[1].view(torch.uint8)[N - 1, 3] = 0xFF
    ws = [K.F8Weight(c, scale()) for c in codes]
    assert [w.plain for w in ws] == [True, False] and not K.F8Weight(codes[0], scale(), "F152").plain
    outs = [torch.full((rows, N), float("nan"), dtype=torch.float16, device="cuda") for _ in ws]
    K.linear(x, ws, outs)
    for c, out in zip(codes, outs):
        p = K.fp8_to_half(c, scale()).double()
        ref, mag = x.double() @ p.T, x.double().abs() @ p.abs().T
        assert ((out.double() - ref).abs() <= 2.0 ** -11 * ref.abs() + (Kd + 2) * 2.0 ** -24 * mag + 2.0 ** -24).all()


# one tile, a number of tiles that is no multiple of sixteen, one that is
@pytest.mark.parametrize("N, Kd", [(16, 128), (40, 200), (264, 4104), (256, 1024)])
def test_every_byte_of_a_tiled_weight_is_written(N, Kd):
    """What a tiled weight holds is no matter of what its buffer held: kernels read the flags behind the tiles in whole words."""
    from poptransformer_amd import _lib
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    codes = torch.randint(1, 120, (N, Kd), dtype=torch.int32, device="cuda").to(torch.uint8)
    buffers = [torch.full((lib.pta_fp8_tiled_bytes(N, Kd),), fill, dtype=torch.uint8, device="cuda") for fill in (0, 0xFF)]
    for b in buffers:
        assert lib.pta_fp8_tile(codes.data_ptr(), b.data_ptr(), N, Kd, 0, stream) == 0
    assert torch.equal(*buffers)
    assert not buffers[1][-(-N // 16) * -(-Kd // 128) * 2048:].any()


@pytest.mark.parametrize("form, M, Kd, N, tiles", [("one", 600, 4096, 2048, "128x128"), ("slices", 1500, 13704, 1032, None), ("pair", 600, 4104, 2048, None), ("one", 2040, 1032, 8192, "256x256")])
def test_channels_beside_the_largest_codes(form, M, Kd, N, tiles):
    """A wave of gemm_block_kernel converts all of its channels one way: those beside a code that the hardware's conversion does not know are bit for bit what they
    are without it, and so is a plain weight in a pair with one that holds such a code.  Weights that are subnormal numbers, which the matrix unit would add with
    fewer bits if they were multiplied as such."""
    from poptransformer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(9)
    n = 2 if form == "pair" else 1
    x = (torch.randn((M, Kd), generator=g, device="cuda") * torch.exp2(torch.randint(-6, 4, (M, Kd), generator=g, device="cuda").float())).half()
    codes = (torch.randint(1, 8, (n, N, Kd), generator=g, device="cuda") | torch.randint(0, 2, (n, N, Kd), generator=g, device="cuda") << 7).to(torch.uint8)
    marked = codes.clone()
    marked[-1, ::32, 5] = 0x7F
    outs = []
    for c in (codes, marked):
        out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
        K.linear(x, [K.F8Weight(w.contiguous(), scale()) for w in c], [out] * n, swiglu=form == "pair", workspace=K.linear_workspace(M, N, "cuda") if form == "slices" else None)
        assert K.linear_kernel() == "gemm_block_kernel" and tiles in (None, K.linear_tiles())
        outs.append(out)
    beside = torch.arange(N, device="cuda") % 32 != 0
    assert torch.equal(outs[0][:, beside], outs[1][:, beside])


def test_a_weight_does_not_wait_for_its_codes():
    """Building one leaves the device at work; a product that is recorded without one before it has the answer as well, or the kernels for all codes, and the same result."""
    from poptransformer_amd import kernels as K
    from poptransformer_amd.engine.loop import recording
    g = torch.Generator(device="cuda").manual_seed(2)
    codes = K.half_to_fp8((torch.randn((520, 1032), generator=g, device="cuda") * 0.02).half(), scale())
    marked = codes.clone()
    marked.view(torch.uint8)[519, 1031] = 0x7F
    x = (torch.randn((3, 1032), generator=g, device="cuda") * 0.2).half()
    outs = [torch.empty((3, 520), dtype=torch.float16, device="cuda") for _ in range(6)]
    K.F8Weight(codes, scale()).plain
    torch.cuda.synchronize()
    torch.cuda._sleep(50_000_000)                 # (some 20 ms, of which building takes a hundredth)
    ws, behind = [K.F8Weight(c, scale()) for c in (codes, marked, codes)], torch.cuda.Event()
    behind.record()
    assert not behind.query()
    host, done = ws[2]._asked
    ws[2]._asked = torch.full((1,), 2, dtype=torch.uint8), done       # (one whose answer is not there)
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with recording(graph, stream=stream):
        for w, out in zip(ws, outs):
            K.linear(x, [w], [out])
    assert [(w._plain, w._asked is None) for w in ws] == [(True, True), (False, True), (False, False)]
    graph.replay()
    ws[2]._asked = host, done
    assert [w.plain for w in ws] == [True, False, True]
    for w, out in zip(ws, outs[3:]):
        K.linear(x, [w], [out])
    assert all(torch.equal(a, b) for a, b in zip(outs, outs[3:])) and torch.equal(outs[0], outs[2]) and not torch.equal(outs[0], outs[1])


def test_copies_know_their_codes():
    """A weight may be copied before a product has asked for the answer."""
    import copy
    from poptransformer_amd import kernels as K
    codes = torch.randint(1, 120, (2, 40, 200), dtype=torch.int32, device="cuda").to(torch.uint8)
    codes[1, 39, 199] = 0xFF
    x = torch.randn((3, 200), device="cuda").half()
    for c, plain in zip(codes, (True, False)):
        copies, out = [f(K.F8Weight(c.contiguous(), scale())) for f in (lambda w: w, copy.copy, copy.deepcopy)], []
        assert all(w.plain is plain for w in copies)
        for w in copies:
            out.append(K.linear(x, [w], [torch.empty((3, 40), dtype=torch.float16, device="cuda")])[0])
        assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])

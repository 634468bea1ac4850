"""The norms' entry points at the edges of what a thread has of a row: one to four pieces of eight columns, whole rows of pieces and a piece more or less."""
import numpy as np
import pytest
import torch

from oracle import ops as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 3])
@pytest.mark.parametrize("cols", [16, 2040, 2048, 2056, 4096, 4104, 6136, 6144, 6152, 8184, 8192])
def test_pieces(rows, cols):
    from poptransformer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(rows + cols)

    def half(*shape):
        return torch.randn(shape, generator=g, device="cuda").half()

    def near(got, ref, ulps):      # (the inverse root and the mean may round to a neighbour by the sums' order)
        got, ref = got.cpu().numpy().astype(np.float32), ref.astype(np.float32)
        assert np.abs(got - ref).max() <= ulps * 2.0 ** -10 * np.abs(ref).max()
    x, gamma, beta, prev, mixes = half(rows, cols), half(cols), half(cols), half(rows, cols), [half(cols) for _ in range(2)]
    hx, hg, hb = (t.cpu().numpy() for t in (x, gamma, beta))
    y = K.rmsnorm(x, gamma, 1e-5)
    near(y, O.rms_norm(hx, hg, 1e-5), 2)
    scale = torch.tensor([-2], dtype=torch.int32, device="cuda")
    for kind in ("F143", "F152"):
        assert torch.equal(K.rmsnorm_fp8_grid(x, gamma, 1e-5, scale, kind), K.half_to_fp8_grid(y, scale, kind))
    if cols >= 8192:
        return
    y = K.layer_norm_ce(x, gamma, beta, 1e-5)
    near(y, O.layer_norm_ce(hx, hg, hb, 1e-5, rows, 1, cols), 4)
    outs, out = [torch.empty_like(x) for _ in mixes], torch.empty_like(x)
    want = [y * w + (1 - w) * prev for w in mixes]
    K.layer_norm_ce_mix(x, gamma, beta, 1e-5, prev, mixes, outs, out=out)
    assert torch.equal(out, y) and torch.equal(prev, y) and all(torch.equal(a, b) for a, b in zip(outs, want))

"""The one-launch iteration of GPT-2 decoders (pta_gpt2_step) against the per-operator path and the oracle."""
import numpy as np
import pytest
import torch

from oracle import models as OM

pytestmark = pytest.mark.gpu


def _cfg(heads, layers=2, vocab=500, positions=700):
    return dict(n_embd=64 * heads, n_head=heads, n_layer=layers, vocab_size=vocab, n_positions=positions, layer_norm_epsilon=1e-5)


def _decoders(cfg, L, B, ffn=None, **kw):
    """Two decoders of the same weights: as one launch, and per operator."""
    from poptransformer_amd.engine import fused, loader
    sd = OM.make_gpt2_state_dict(cfg, seed=3)
    rng = np.random.default_rng(5)
    for k in sd:                          # biases and norms that a wrong index would show
        if k.endswith("bias"):
            sd[k] = rng.normal(0, 0.05, sd[k].shape).astype(np.float16)
        elif "ln_" in k:
            sd[k] = rng.normal(1, 0.1, sd[k].shape).astype(np.float16)
    if ffn is not None:
        for i in range(cfg["n_layer"]):
            p = f"transformer.h.{i}.mlp."
            sd[p + "c_fc.weight"], sd[p + "c_fc.bias"] = sd[p + "c_fc.weight"][:ffn], sd[p + "c_fc.bias"][:ffn]
            sd[p + "c_proj.weight"] = np.ascontiguousarray(sd[p + "c_proj.weight"][:, :ffn])
    weights = loader.gpt2_weights(sd, cfg)
    one, per_op = (fused.FusedDecoder(loader.gpt2_spec(cfg, L, B, 0, kw.get("eos", 1), kw.get("early_stop", False)), weights) for _ in range(2))
    assert one.chained is not None
    per_op.chained = None
    return one, per_op


def _close(a, b):
    """Logits of two paths that differ by the order of fp32 sums: roundings to fp16 between two layers, 2^-11 each and some ten of them a layer."""
    d, n = (a.float() - b.float()).norm().item(), b.float().norm().item()
    assert np.isfinite(d) and d <= 0.006 * n, (d, n)


@pytest.mark.parametrize("heads,B,ffn,L", [(1, 1, None, 24), (1, 3, 72, 24), (3, 2, None, 40), (4, 1, 1016, 24), (4, 8, None, 24), (5, 5, None, 24),
                                           (12, 1, None, 40), (12, 4, None, 24), (20, 1, None, 24), (20, 8, None, 24), (25, 2, None, 24), (32, 1, None, 24)])
def test_one_launch_follows_the_per_operator_path(heads, B, ffn, L):
    one, per_op = _decoders(_cfg(heads), L, B, ffn)
    ids = np.zeros((B, L), np.int32)
    ids[:, :] = np.random.default_rng(heads).integers(2, 500, size=(B, L))
    for d in (one, per_op):
        d.reset(ids)
    for _ in range(L - 1):                # the tokens are given: each step's logits are compared
        one.step_fn()
        per_op.step_fn()
        _close(one.logits, per_op.logits)
        assert torch.equal(one.next_ids.cpu(), one.logits.float().argmax(1).int().cpu())
    torch.cuda.synchronize()
    assert not one.chained.failed()
    assert int(one.step.item()) == L - 1 and torch.equal(one.container, per_op.container) and torch.equal(one.mask, per_op.mask)
    for a, b in zip(one.rings, per_op.rings):
        assert (a.float() - b.float()).norm() <= 0.006 * b.float().norm()


@pytest.mark.parametrize("B", [1, 4])
def test_contexts_of_several_visits_and_a_ring_that_comes_round(B):
    one, per_op = _decoders(_cfg(2, layers=1, positions=610), 600, B)
    ids = np.random.default_rng(1).integers(2, 500, size=(B, 600)).astype(np.int32)
    for d in (one, per_op):
        d.reset(ids)
        d.consume_prompt(250)
    for _ in range(14):                   # contexts 250 .. 263: a second visit of 256 rows begins
        one.step_fn(), per_op.step_fn()
        _close(one.logits, per_op.logits)
    for d in (one, per_op):
        d.reset(ids)
        d.consume_prompt(597)
    for _ in range(8):                    # positions 597 .. 604: the last five in places of the ring that had others
        one.step_fn(), per_op.step_fn()
        _close(one.logits, per_op.logits)


@pytest.mark.parametrize("B,early_stop", [(1, True), (3, False)])
def test_generated_tokens_equal_the_oracle(B, early_stop):
    """Tokens of the oracle's loop, end tokens, early stop and the recorded iteration's replays included."""
    from poptransformer_amd.engine import fused, loader
    cfg, L, pad = _cfg(4), 20, 0
    sd = OM.make_gpt2_state_dict(cfg, seed=11)
    ids = np.zeros((B, L), np.int32)
    ids[:, :4] = np.random.default_rng(0).integers(3, 500, size=(B, 4))
    free, _ = OM.run_decode_loop(OM.GPT2Oracle(sd, cfg, L, B), ids, L, L - 1, pad, 499)
    eos = int(free[0, 9])                 # a token that the first sequence reaches
    ref_c, ref_s = OM.run_decode_loop(OM.GPT2Oracle(sd, cfg, L, B), ids, L, L - 1, pad, eos, early_stop=early_stop)
    dec = fused.FusedDecoder(loader.gpt2_spec(cfg, L, B, pad, eos, early_stop), loader.gpt2_weights(sd, cfg))
    dec.capture()
    for _ in range(2):
        got_c, got_s = dec.run(ids, L - 1, check_every=1)
        assert dec.chained is not None and got_s == ref_s and np.array_equal(got_c, ref_c)


def test_iterations_of_two_decoders_at_once():
    """Launches on two streams share the machine: each waits only for workgroups that have started before."""
    pairs = [_decoders(_cfg(12, layers=3), 40, 1), _decoders(_cfg(4, layers=6), 40, 4)]
    ids = [np.random.default_rng(i).integers(2, 500, size=(d[0].spec.batch, 40)).astype(np.int32) for i, d in enumerate(pairs)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for (one, per_op), i in zip(pairs, ids):
        one.reset(i), per_op.reset(i)
    torch.cuda.synchronize()
    for _ in range(30):
        for (one, _), s in zip(pairs, streams):
            with torch.cuda.stream(s):
                one.step_fn()
    torch.cuda.synchronize()
    for one, per_op in pairs:
        per_op.run_steps(30)
        assert not one.chained.failed()
        _close(one.logits, per_op.logits)


def test_shapes_and_options_that_stay_per_operator():
    from poptransformer_amd import kernels as K
    from poptransformer_amd.engine import fused, loader
    cfg = _cfg(4)
    w = loader.gpt2_weights(OM.make_gpt2_state_dict(cfg, seed=3), cfg)

    def made(weights=w, **kw):
        spec = loader.gpt2_spec(cfg, 24, kw.pop("B", 1), 0, 1)
        for k, v in kw.items():
            setattr(spec, k, v)
        return fused.FusedDecoder(spec, weights).chained
    assert made() is not None and made(B=8) is not None
    assert made(B=9) is None and made(topk=4) is None and made(fp8_cache=True) is None and made(max_len=701) is None
    one = made()
    assert isinstance(one, K.Gpt2Step) and not one.failed()


def test_tensors_that_are_not_what_the_spec_says_stay_per_operator():
    """What the operators refuse is refused, and what they take is computed as they do."""
    import dataclasses
    from poptransformer_amd import kernels as K
    from poptransformer_amd.engine import fused, loader
    cfg = _cfg(4)
    w = loader.gpt2_weights(OM.make_gpt2_state_dict(cfg, seed=3), cfg)
    ids = np.random.default_rng(2).integers(2, 500, size=(2, 24)).astype(np.int32)
    ids[:, 0] = 450, 7

    def made(**kw):
        dec = fused.FusedDecoder(loader.gpt2_spec(cfg, 24, 2, 0, 1), dataclasses.replace(w, **kw))
        dec.reset(ids)
        assert dec.chained is None
        return dec

    def block(**kw):
        return [w.blocks[0], dataclasses.replace(w.blocks[1], **kw)]
    b, d = w.blocks[1], w.embed.shape[1]
    narrow = fused.LinearWeights(K.F16Weight(torch.zeros((d, d - 64), dtype=torch.float16, device="cuda")), b.out.bias)
    wide = torch.zeros((w.embed.shape[0], 2 * d), dtype=torch.float16, device="cuda")
    wide[:, ::2] = w.embed
    for kw in (dict(embed=w.embed.float()), dict(embed=wide[:, ::2]), dict(blocks=block(out=narrow)), dict(blocks=block(mlp_out=narrow))):
        with pytest.raises(ValueError):
            made(**kw).step_fn()
    # a table of fewer tokens than the head has: ids past its end are its last row's
    short, last = made(embed=w.embed[:400].contiguous()), fused.FusedDecoder(loader.gpt2_spec(cfg, 24, 2, 0, 1), w)
    last.reset(np.minimum(ids, 399))
    last.chained = None
    for dec in (short, last):
        dec.step_fn()
    assert torch.equal(short.logits, last.logits)
    # (no result of these is looked at: the operators do not check them either)
    made(pos_embed=w.pos_embed.float()), made(blocks=block(norm1=(b.norm1[0].float(), b.norm1[1]))), made(final_norm=(w.final_norm[0], w.final_norm[1][:-8].clone()))
    made(blocks=block(qkv=[fused.LinearWeights(K.F16Weight(torch.zeros((2 * d, d), dtype=torch.float16, device="cuda")), b.qkv[0].bias)]))
    made(blocks=block(out=fused.LinearWeights(b.out.w, b.out.bias.float())))


@pytest.mark.parametrize("clear", ["all", "word"])
def test_a_wait_that_gave_up_is_reported_and_cleared(clear):
    """The word that a wait sets when it gives up, set by hand, where words of the next iteration's number lie about: launches do nothing, `run` raises, and
    once cleared - by the decoder, or the word alone behind a launch that found it - no such word is taken for one that has arrived."""
    one, per_op = _decoders(_cfg(4), 24, 2)
    ids = np.random.default_rng(4).integers(2, 500, size=(2, 24)).astype(np.int32)
    per_op.run(ids, 12)
    for graph in (False, True):
        if graph:
            one.capture()
        one.run(ids, 3)
        words = one.chained.workspace.view(torch.int32)
        assert int(words[0]) == 0 and int(words[1]) == 0
        words[64:] = (int(words[2]) + 1 & 0xFFFF) << 16 | 0x3C00                  # ones that seem to have arrived
        words[1] = 1
        torch.cuda.synchronize()
        with pytest.raises(RuntimeError, match="clear_failure"):
            one.run(ids, 3)
        assert int(one.step.item()) == 0
        if clear == "all":
            one.chained.clear_failure()
        else:
            words[1] = 0
            torch.cuda.synchronize()
        got, step = one.run(ids, 12)
        assert step == 12
        _close(one.logits, per_op.logits)


@pytest.mark.parametrize("B", [1, 2, 3, 8])
def test_norms_are_those_of_the_operators(B):
    """A key projection that hands the normed row on: the ring then holds the norms' results, bit for bit those of layer_norm_ce.  Rows of small multiples of
    1/16 with mean 0, whose sums are the same in any order; their squares add up to numbers whose reciprocal root lies so near the middle of two fp16
    numbers that the hardware's own (v_rsq_f32) falls on the other side of it."""
    from poptransformer_amd import kernels as K
    from poptransformer_amd.engine import fused, loader
    squares = [17680, 21316, 114192, 147636, 295638, 296560, 302818, 312250, 505720, 521874, 621112, 626752, 643156, 653108, 672664, 693112, 798424, 883610, 899668,
               963054, 1027398, 1058372, 1111148, 1136136, 1216374, 1292714, 1302582, 1328482, 1423866, 1461878, 1468644, 1508476, 1604728, 1695658, 1767344, 1771834]
    L, d = 72, 64
    cfg = _cfg(1, layers=1, vocab=2 + 2 * len(squares), positions=L)
    sd, rng = OM.make_gpt2_state_dict(cfg, seed=3), np.random.default_rng(8)
    table = np.zeros((cfg["vocab_size"], d))
    for token in range(2, len(table)):
        rest, half = squares[(token - 2) % len(squares)] // 2, []
        while rest:
            half.append(min(int(np.sqrt(rest)), 255))
            rest -= half[-1] ** 2
        row = np.zeros(d)
        row[:2 * len(half)] = half + [-v for v in half]
        table[token] = rng.permutation(row) / 16
    a, n = "transformer.h.0.attn.c_attn.", "transformer.h.0.ln_1."
    for key, value in {"transformer.wte.weight": table, "transformer.wpe.weight": np.zeros((L, d)), a + "weight": np.concatenate([np.zeros((d, d)), np.eye(d), np.eye(d)]),
                       a + "bias": np.zeros(3 * d), n + "weight": np.ones(d), n + "bias": np.zeros(d)}.items():
        sd[key] = value.astype(np.float16)
    dec = fused.FusedDecoder(loader.gpt2_spec(cfg, L, B, 0, 1), loader.gpt2_weights(sd, cfg))
    ids = np.stack([rng.permutation(np.arange(2, 2 + L)) for _ in range(B)]).astype(np.int32)
    dec.reset(ids)
    for _ in range(L):
        dec.step_fn()
    torch.cuda.synchronize()
    assert dec.chained is not None and not dec.chained.failed()
    x = torch.from_numpy(sd["transformer.wte.weight"][ids]).cuda()
    gamma, beta = torch.ones(d, dtype=torch.float16, device="cuda"), torch.zeros(d, dtype=torch.float16, device="cuda")
    want = torch.stack([K.layer_norm_ce(x[:, t].contiguous(), gamma, beta, cfg["layer_norm_epsilon"]) for t in range(L)], 1)
    for got in dec.rings[0].reshape(2, B, L, d):                                  # keys, values
        differ = (got != want).any(2).sum().item()
        assert differ == 0, differ


def test_caches_of_several_thousand_positions_stay_per_operator():
    from poptransformer_amd.engine import fused, loader
    cfg = _cfg(1, layers=1, positions=5000)
    w = loader.gpt2_weights(OM.make_gpt2_state_dict(cfg, seed=3), cfg)
    assert [fused.FusedDecoder(loader.gpt2_spec(cfg, n, 1, 0, 1), w).chained is not None for n in (4096, 4097, 5000)] == [True, False, False]

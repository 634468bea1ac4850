"""The prompt in passes of several positions.

The reference's GPT-2, Llama-2 and ChatGLM2 loops take a prompt one position per iteration: the
container already holds the prompt's tokens, so the token an iteration selects is dropped and the
stored one is used (models/base_model.py:313-318).  Those iterations only fill the KV cache.  Its
two-stage ChatGLM model runs the same layer stack once over the whole prompt with sequence_length > 1
(models/chatglm/model.py:301-330, models/chatglm/attention.py:89-140) before the loop starts.

`PromptPass` is that first stage for the decoders here: R consecutive positions of every sequence
(B*R <= 2048 rows) go through each layer together - the projections as GEMMs over B*R rows, which read
each weight once per pass, the rotary embedding and cache append per row at its own position, and
causal attention of row r over positions 0..p0+r.  The final norm, the head and the token selection
are skipped: the loop would discard their result.  What it leaves in the KV rings is what R iterations
of the loop leave there, up to the rounding of a different summation order in the GEMMs.
"""
from collections import OrderedDict

import torch

from .. import _lib
from .. import kernels as K
from .fused import LayerOps
from .loop import recording


class RowMemory:
    """The row buffers of all passes of up to `rows` rows: each pass takes the first rows of every buffer, in the same order.  Passes follow each other on one
    stream, and none looks at what another has left."""

    def __init__(self, rows, device):
        self.rows, self.device, self.made = rows, device, []

    def taken(self):
        """The buffers from the first one on, for one pass."""
        return RowBuffers(self)


class RowBuffers:
    def __init__(self, memory):
        self.memory, self.next = memory, 0

    def _next(self, make):
        if self.next == len(self.memory.made):
            self.memory.made.append(make(self.memory.rows))
        self.next += 1
        return self.memory.made[self.next - 1]

    def buffer(self, rows, *shape, dtype=torch.float16):
        t = self._next(lambda n: torch.empty((n, *shape), dtype=dtype, device=self.memory.device))
        if t.shape[1:] != shape or t.dtype != dtype or rows > len(t):
            raise RuntimeError(f"prompt pass: buffer [{rows}, {shape}] {dtype} where others have {tuple(t.shape)} {t.dtype}")
        return t[:rows].zero_()

    def scratch(self, make, rows):
        """make(rows): the bytes that so many rows need."""
        return self._next(make)


class PromptPasses:
    """The passes of a decoder by their number of positions, those used last.  They share row buffers (at the 7B width, 2048 rows with a cache of 2048: 2 GB,
    which each length of prompts would hold for itself else): a pass takes the smallest set that has its rows.  The first set is as large as its pass needs, a
    larger one that is needed later at least half as large again, so that all of them together stay below four times the largest pass's.  Recorded passes take
    what else they need from one pool."""

    most_rows, most = 2048, 256      # of a pass; passes that are kept

    def __init__(self, dec):
        self.dec, self.memory, self.passes, self.pool = dec, [], OrderedDict(), None

    def _memory(self, rows):
        fit = [m for m in self.memory if m.rows >= rows]
        if not fit:
            largest = max((m.rows for m in self.memory), default=0)
            fit.append(RowMemory(max(rows, min(self.most_rows, largest * 3 // 2)), self.dec.dev))
            self.memory += fit
        return min(fit, key=lambda m: m.rows)

    def of(self, rows):
        if rows not in self.passes:
            while len(self.passes) >= self.most:
                torch.cuda.current_stream().synchronize()      # (a replay may be on its way)
                self.passes.popitem(last=False)
            if self.pool is None:
                self.pool = torch.cuda.graph_pool_handle()
            self.passes[rows] = PromptPass(self.dec, rows, self._memory(self.dec.spec.batch * rows).taken(), self.pool)
        self.passes.move_to_end(rows)
        return self.passes[rows]


class PromptPass(LayerOps):
    """One pass over the layers of B*rows rows; shares weights and KV rings with the decoder `dec`, row buffers with its other passes."""

    def __init__(self, dec, rows, memory, pool):
        super().__init__(dec.spec, dec.w, dec.dev, dec.spec.batch * int(rows), memory)
        self.dec, self.rows, self.pool = dec, int(rows), pool
        s, i32 = self.spec, torch.int32
        self.first = torch.zeros((), dtype=i32, device=self.dev)       # position of row 0 of every sequence
        self._offsets = torch.arange(self.rows, dtype=i32, device=self.dev)
        self.graph = None
        if self._lin_ws is None:
            self._lin_ws = self._linear_workspace(s.d_model, self.w.blocks[0].mlp_out.K)

    def _linear_workspace(self, d, ffn):
        """Scratch for the K split of the projections with few output channels (attention output, MLP down): what this pass's rows need of the shared one, so
        that a product is cut alike whatever passes there were."""
        shared = self._scratch(lambda n: K.linear_workspace(n, max(d, ffn), self.dev), self._rows)
        return shared[:K.linear_workspace_bytes(self._rows, max(d, ffn))]

    def run(self, p0):
        """Positions p0 .. p0+rows-1 of every sequence (row b*rows + r is sequence b at p0 + r).  The pass
        depends on device state only (`first`, the container, the rings): the first call runs it eagerly,
        the second records it into a HIP graph, later calls replay that graph."""
        s = self.spec
        if p0 < 0 or p0 + self.rows > s.max_len:
            raise ValueError(f"prompt pass over positions {p0}..{p0 + self.rows - 1} leaves the cache (max_len {s.max_len})")
        self.first.fill_(p0)
        if self.graph is not None:
            self.graph.replay()
        elif not getattr(self, "_warm", False):
            self._layers()
            self._warm = True
        else:
            stream = torch.cuda.current_stream()
            stream.synchronize()
            self.graph = torch.cuda.CUDAGraph()
            with recording(self.graph, pool=self.pool, stream=stream):
                self._layers()
            self.graph.replay()

    def _layers(self):
        s, w, dec = self.spec, self.w, self.dec
        B, R = s.batch, self.rows
        positions = self._offsets + self.first
        ids = dec.container.index_select(1, positions).reshape(-1)
        K.embedding(w.embed, ids, self.x)
        if w.pos_embed is not None:        # GPT-2: learned positions, one table row per position
            self.x.add_(w.pos_embed.index_select(0, positions).repeat(B, 1))
        h, nrm = self._normed(self.x, w.blocks[0].norm1, w.blocks[0].qkv)
        for li, blk in enumerate(w.blocks):
            if not hasattr(self, "_qkv_views"):
                self._prepare_qkv_views(blk)
            self._linear_group(h, blk.qkv, self._qkv_bufs, nrm)
            qp, kp, vp, qs, ks, vs = self._qkv_views
            K.prompt_rope_append(qp, kp, vp, self.q_rot, dec.rings[li], self.first, w.inv_freq, B, R, s.n_head,
                                 s.n_kv_head, s.head_dim, s.max_len, s.rope, qs, ks, vs, kv_scale=dec.kv_scale)
            K.prompt_attention(self.q_rot, dec.rings[li], self.first, self.attn_ws, self.ctx, B, R, s.n_head,
                               s.n_kv_head, s.head_dim, s.max_len, s.scale_scores, kv_scale=dec.kv_scale)
            h, nrm = self._added_and_normed(self.ctx, blk.out, blk.norm2, blk.mlp_in)
            if len(blk.mlp_in) == 2:
                self._linear_group(h, blk.mlp_in, [self.act, self.act], nrm, swiglu=True, consumer=blk.mlp_out)
            else:
                self._linear(h, blk.mlp_in[0], self.act, act=_lib.ACT_GELU_TANH, norm=nrm)
            if li + 1 < len(w.blocks):
                h, nrm = self._added_and_normed(self.act, blk.mlp_out, w.blocks[li + 1].norm1, w.blocks[li + 1].qkv)
            else:
                self._linear(self.act, blk.mlp_out, self.x, residual=self.x)

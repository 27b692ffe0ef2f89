"""A decode step's layers in one launch, for models whose every layer is the same pre-norm block of
grouped-query attention and SwiGLU (`src/model/layers/rmsnorm_gqa_swiglu_block.zig:10-51`)."""
from __future__ import annotations

import torch

from .. import ops
from ..ops import decode_layers as kernel
from ..parts.attention import GqaAttention
from ..parts.block import PreNormBlock
from ..parts.mlp import SwiGluMlp
from ..parts.norm import GivenRmsNorm, RmsNorm


STATUS = "one_launch.status"      # of an engine's kept buffers: 1 once a wait has come to its end


class OneLaunchLayers:
    """What the kernel takes of a bound ``DecoderModel``, and its launch.  (The model owns this and
    is handed in: a reference back would keep both, and the weights, until the collector runs.)"""

    def __init__(self, model):
        a = model.blocks[0].mixer.spec
        self.ff = model.blocks[0].feed_forward.spec.intermediate_size
        self.hidden = model.spec.hidden_size
        self.heads, self.kv_heads = a.n_heads, a.n_kv_heads
        self.tables = model.blocks[0].mixer.position.rotation_tables()
        index = torch.device(model.ctx.device).index or 0
        self.wgs, self.cus = kernel.workgroups(index), kernel.compute_units(index)

    @staticmethod
    def of(model):
        """For ``model`` once its weights are bound, or None where it is of another kind."""
        s, blocks = model.spec, model.blocks
        if model.ctx.compute_dtype != torch.bfloat16 or torch.device(model.ctx.device).type != "cuda" \
                or not blocks or s.streams is not None or s.position_table_name is not None \
                or s.sinusoidal_positions is not None or s.embedding_norm is not None \
                or model.reentry is not None or type(model.final_norm) is not RmsNorm \
                or len(s.schedule) != len(blocks) \
                or any(e.layer != i or e.cache_of is not None or e.reentry
                       for i, e in enumerate(s.schedule)):
            return None
        first = blocks[0]
        for b in blocks:
            if type(b) is not PreNormBlock or type(b.mixer) is not GqaAttention \
                    or type(b.feed_forward) is not SwiGluMlp or type(b.mixer_norm) is not RmsNorm \
                    or type(b.ff_norm) is not RmsNorm:
                return None
            m, f = b.mixer, b.feed_forward
            if not (m.qkv.tiled and m.o.tiled and f.fused and f.gate_up.tiled and f.down.tiled) \
                    or m.spec != first.mixer.spec or f.spec != first.feed_forward.spec \
                    or m.spec.window is not None or m.position.custom_apply \
                    or b.mixer_norm.spec.eps != first.mixer_norm.spec.eps \
                    or b.ff_norm.spec.eps != first.ff_norm.spec.eps \
                    or any(t is not None and t.data_ptr() % 16 != 0 for t in
                           (m.q_gain, m.k_gain, b.ff_norm.gain, b.mixer_norm.gain)):
                return None
        if model.final_norm.gain.data_ptr() % 16 != 0:
            return None
        return OneLaunchLayers(model)

    def takes(self, model, step, caches, given) -> bool:
        """Whether this step runs here: a token a sequence, with what the first norm needs of the
        stream's rows already made (``given``).  Not where classes of kernels are measured, each alone or
        all together: the layers' one launch is of no class."""
        if step.max_q_len != 1 or model.layer_probe is not None or ops.measures_classes() \
                or not isinstance(given, GivenRmsNorm):
            return False
        cache = caches[0]
        keys = step.kv_tables(cache.group).max_pages * cache.page_size
        if keys > kernel.MAX_CONTEXT or not kernel.pays(step.n_tokens, self.hidden, self.ff, self.heads,
                                                        self.kv_heads, keys, self.cus):
            return False
        if not kernel.sizes_covered(step.n_tokens, self.hidden, self.ff, self.heads, self.kv_heads,
                                    model.blocks[0].mixer.spec.head_dim, cache.page_size, self.wgs):
            return False
        return all(c.writes and c.group == cache.group and c.page_size == cache.page_size
                   and c.k_pool.dtype == c.v_pool.dtype == torch.bfloat16 for c in caches)

    @staticmethod
    def _table(model, step, caches) -> torch.Tensor:
        """The layers' records on the device, made once an engine."""
        blocks = model.blocks
        norms = [b.mixer_norm for b in blocks[1:]] + [model.final_norm]
        records = (kernel.Layer * len(blocks))()
        at = lambda t: None if t is None else t.data_ptr()
        for r, b, c, after in zip(records, blocks, caches, norms):
            m, f = b.mixer, b.feed_forward
            r.w[:] = [at(x.weight) for x in (m.qkv, m.o, f.gate_up, f.down)]
            r.q_gain, r.k_gain, r.ff_gain, r.next_gain = (
                at(t) for t in (m.q_gain, m.k_gain, b.ff_norm.gain, after.gain))
            r.k_pool, r.v_pool = at(c.k_pool), at(c.v_pool)
        raw = bytes(records)
        return step.made("decode_layers." + raw.hex(), lambda device: torch.frombuffer(
            bytearray(raw), dtype=torch.uint8).to(device))

    def forward(self, model, step, caches, x, given):
        """Every layer over ``x`` in place; returns what is left for the final norm."""
        b, cache = model.blocks[0], caches[0]
        eps = b.mixer.spec.qk_norm_eps
        kv = step.kv_tables(cache.group)
        cos, sin = self.tables if self.tables is not None else (None, None)
        M = x.shape[0]
        words = step.made(f"decode_words.{M}", lambda device: kernel.words(
            M, self.hidden, self.ff, self.heads, self.kv_heads, device))
        status = step.made(STATUS, lambda device: torch.zeros((1,), dtype=torch.int32, pin_memory=True))
        kernel.decode_layers(
            self._table(model, step, caches), len(caches), x, given.xg, given.sq, self.ff, self.heads,
            self.kv_heads, cache.page_size, float(b.mixer_norm.spec.eps), float(b.ff_norm.spec.eps),
            0.0 if eps is None else float(eps), float(b.mixer.scale), cos, sin, step.positions,
            kv.slot_mapping, kv.block_table, step.ctx_len, words, status)
        return GivenRmsNorm(model.final_norm, x, given.xg, given.sq)

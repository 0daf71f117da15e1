"""Prompt steps of decoders made of like dense layers, a layer launched by one call.

A layer of such a decoder is nine launches; made one by one through the parts they cost more than a step of up to a
few hundred rows takes to run.  The kernel library makes the same launches in the same order (``sb_dense_layers``), so
the results have the same bits; the parts remain the description of the model and the way everything else runs:
decode steps (recorded once and replayed), traced steps, choices imposed on the launchers, layers of any other kind.
"""
from __future__ import annotations

from typing import Optional

import torch

from .. import ops
from ..parts.attention import Attention
from ..parts.block import PreNormBlock
from ..parts.ffn import GatedDenseFFN
from ..parts.norm import RMSNorm

# Where the launches are the longer part of a step: rows times a layer's weights, and the weights alone, whose reading takes
# longer than nine launches from Python (86 us) past some 100 M.  Steps of random tokens, part by part against a call a layer (us,
# each waited for): 0.5B sizes (15 M weights a layer) 288 rows 2,285 and 1,716, 512 rows 2,280 and 2,150, 640 rows 2,614 and
# 2,638; 1.5B sizes (47 M) 128 rows 2,618 and 2,412, 183 rows 2,614 and 2,625 (one step after another 2,494 and 2,385), 288 rows 2,944
# and 3,031; 3B sizes (77 M) 65 rows 3,348 and 3,091, 128 rows 3,383 and 3,445; 7B sizes (233 M) 2 rows 3,285 and 3,308.
# Layers 256 wide gain at every count of rows measured (1,536: 2,398 and 2,167), and more were not.
MAX_WORK = 8.6e9
MAX_WEIGHTS = 100e6
MAX_ROWS = 1536


_DTYPES = {torch.float32: 0, torch.bfloat16: 1}


def _plain_norm(norm) -> bool:
    return type(norm) is RMSNorm and norm.groups == 1 and norm.offset == 0.0 and norm.weight is not None


def _takes(block, first, rt) -> bool:
    """Whether the block is such a layer, of the sizes of ``first``."""
    if type(block) is not PreNormBlock or block.input_conv is not None or type(block.ffn) is not GatedDenseFFN:
        return False
    m, f = block.mixer, block.ffn
    if type(m) is not Attention or m.extended or m.out_scale != 1.0 or f.out_scale != 1.0 or not (
            _plain_norm(block.mixer_norm) and _plain_norm(block.ffn_norm)):
        return False
    tables = m.position.rotary_tables()
    if tables is None or m.position.interleaved or getattr(m.position, "magnitude", 1.0) != 1.0:
        return False
    if any(p.packed is None for p in (m.qkv, m.out, f.gate_up, f.down)) or m.out.bias is not None or f.down.bias is not None:
        return False
    if m.qkv.bias is not None and m.qkv.bias.dtype != torch.float32:
        return False
    g, w = first.mixer, first.ffn
    return (m.width, m.heads_q, m.heads_kv, m.head_dim, f.inner, m.row_tile) == (g.width, g.heads_q, g.heads_kv, g.head_dim, w.inner, g.row_tile)


def takes_step(ctx) -> bool:
    """Whether a step is one whose launches may be made in one call a layer."""
    return not ctx.is_decode and ctx.n_rows <= MAX_ROWS and ops.launchers_choose()


class DenseLayers:
    """The like layers of a model, launched by one call each.  A layer is looked at, and its addresses are gathered, when its
    turn comes in a step (some 3 us): nothing is held that may have been exchanged since, and the GPU has the layers before it
    to work on meanwhile.  (With all layers gathered ahead of the first launch a step lost 0.1 ms, up to 5 % where its kernels
    are the longer part.)"""

    @classmethod
    def of(cls, model, bindings) -> Optional["DenseLayers"]:
        rt = model.rt
        if not rt.fast_kernels or rt.act_dtype != torch.bfloat16 or rt.cache_dtype != torch.bfloat16 or model.junctions or not model.order:
            return None
        run = cls(model, bindings)
        return run if run.takes(0) and ops.attention_mfma_ok(torch.bfloat16, torch.bfloat16, run.first.mixer.head_dim) else None

    def __init__(self, model, bindings):
        self.model, self.bindings = model, bindings
        self.first = model.blocks[model.order[0].block]
        self.step = None

    def pays(self, rows: int) -> bool:
        """Whether the launches of a step of ``rows`` rows are its longer part."""
        m, f = self.first.mixer, self.first.ffn
        weights = sum(p.rows * p.n_in for p in (m.qkv, m.out, f.gate_up, f.down))
        return weights <= MAX_WEIGHTS and rows * weights <= MAX_WORK

    def takes(self, i: int) -> bool:
        """Whether entry ``i`` of the run order is a layer like the first."""
        e, b, first = self.model.order[i], self.bindings[i], self.bindings[0]
        return _takes(self.model.blocks[e.block], self.first, self.model.rt) and e.junction is None and b.writes_cache \
            and b.group == first.group and b.k_cache.dtype == torch.bfloat16

    def layer(self, i: int, x: torch.Tensor, ctx, h: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
        """Entry ``i`` on the stream ``x`` in place; ``h`` its norm of ``x`` if the entry before has left it.  Returns the next
        entry's norm of ``x``, where that is one the last kernel applies."""
        order, bind = self.model.order, self.bindings[i]
        block = self.model.blocks[order[i].block]
        m, f, L = block.mixer, block.ffn, ops.DenseLayer()
        inv_freq, factors, rot = m.position.rotary_tables()
        L.qkv_w, L.out_w = m.qkv.packed.data_ptr(), m.out.packed.data_ptr()
        L.gate_up_w, L.down_w = f.gate_up.packed.data_ptr(), f.down.packed.data_ptr()
        L.qkv_bias = None if m.qkv.bias is None else m.qkv.bias.data_ptr()
        norm = block.ffn_norm
        L.norm_w, L.norm_dtype, L.norm_eps = norm.weight.data_ptr(), _DTYPES[norm.weight.dtype], norm.eps
        norm = getattr(self.model.blocks[order[i + 1].block], "first_norm", None) if i + 1 < len(order) else None
        follows = _plain_norm(norm)
        if follows:
            L.next_w, L.next_dtype, L.next_eps = norm.weight.data_ptr(), _DTYPES[norm.weight.dtype], norm.eps
        L.inv_freq = None if inv_freq is None else inv_freq.data_ptr()
        L.freq_factors = None if factors is None else factors.data_ptr()
        L.rot_dims, L.window, L.scale = rot, m.window, m.scale
        L.gate = ops.gate_code(f.activation)
        L.k_cache, L.v_cache = bind.k_cache.data_ptr(), bind.v_cache.data_ptr()
        if h is None:
            h = block.mixer_norm.forward(x, torch.bfloat16)
        if self.step is None:
            height = ops.attention_tile_height(ctx, m.heads_q, m.heads_kv, m.row_tile)
            self.step = ops.DenseStep(x, f.inner, m.heads_q, m.heads_kv, m.head_dim, ctx.page_table(bind.group), bind.k_cache.shape[0],
                                      ctx.row_pos, ctx.row_seq, ctx.row_tiles(height), height,
                                      ops.attention_row_groups(ctx, height, m.heads_q))
        self.step.run(L, h)
        return h if follows else None

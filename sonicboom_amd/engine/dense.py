"""Prompt steps of decoders made of like dense layers, with all layers launched by one call.

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

# Rows up to which the launches are the longer part of a step (0.5B sizes: 2.1 ms of launches a step against
# 1.5 ms of kernels at 288 rows and some 3 ms at 1,500; larger sizes cross earlier).
MAX_ROWS = 1536


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
    """Whether a step is one whose launches are worth making in one call, and free to be."""
    return not ctx.is_decode and ctx.n_rows <= MAX_ROWS and ops.launchers_choose()


class DenseLayers:
    """The layers of a model that is nothing but a run of them, with the addresses that the library takes.  Made anew for
    every step (some 150 us for 28 layers): it holds no address of a part that may have been exchanged since."""

    @classmethod
    def of(cls, model, bindings) -> Optional["DenseLayers"]:
        rt = model.rt
        if not rt.fast_kernels or rt.act_dtype != torch.bfloat16 or rt.cache_dtype != torch.bfloat16 or model.junctions or not model.order:
            return None
        blocks = [model.blocks[e.block] for e in model.order]
        for block, e, b in zip(blocks, model.order, bindings):
            if not _takes(block, blocks[0], rt) or e.junction is not None or not b.writes_cache or b.group != bindings[0].group \
                    or b.k_cache.dtype != torch.bfloat16:
                return None
        if not ops.attention_mfma_ok(torch.bfloat16, torch.bfloat16, blocks[0].mixer.head_dim):
            return None
        return cls(blocks, bindings)

    def __init__(self, blocks, bindings):
        self.first, self.group = blocks[0], bindings[0].group
        self.n_pages = bindings[0].k_cache.shape[0]
        self.layers = (ops.DenseLayer * len(blocks))()
        dt = {torch.float32: 0, torch.bfloat16: 1}
        for i, (block, bind) in enumerate(zip(blocks, bindings)):
            m, f, L = block.mixer, block.ffn, self.layers[i]
            inv_freq, factors, rot = m.position.rotary_tables()
            L.qkv_w, L.out_w = m.qkv.packed.data_ptr(), m.out.packed.data_ptr()
            L.gate_up_w, L.down_w = f.gate_up.packed.data_ptr(), f.down.packed.data_ptr()
            L.qkv_bias = None if m.qkv.bias is None else m.qkv.bias.data_ptr()
            norm = block.ffn_norm
            L.norm_w, L.norm_dtype, L.norm_eps = norm.weight.data_ptr(), dt[norm.weight.dtype], norm.eps
            if i + 1 < len(blocks):
                norm = blocks[i + 1].mixer_norm
                L.next_w, L.next_dtype, L.next_eps = norm.weight.data_ptr(), dt[norm.weight.dtype], norm.eps
            L.inv_freq = None if inv_freq is None else inv_freq.data_ptr()
            L.freq_factors = None if factors is None else factors.data_ptr()
            L.rot_dims, L.window, L.scale = rot, m.window, m.scale
            L.gate = ops.gate_code(f.activation)
            L.k_cache, L.v_cache = bind.k_cache.data_ptr(), bind.v_cache.data_ptr()

    def __call__(self, x: torch.Tensor, ctx) -> None:
        """All layers on the stream ``x`` in place."""
        m = self.first.mixer
        h = self.first.mixer_norm.forward(x, torch.bfloat16)
        height = ops.attention_tile_height(ctx, m.heads_q, m.heads_kv, m.row_tile)
        ops.dense_layers(x, h, self.layers, self.first.ffn.inner, m.heads_q, m.heads_kv, m.head_dim, ctx.page_table(self.group),
                         self.n_pages, ctx.row_pos, ctx.row_seq, ctx.row_tiles(height), height)

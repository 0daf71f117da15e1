"""Latent-attention layers with heads of 128 + 64 numbers and 128 values, whose prompt steps may build keys and values: the layer
against 64-bit arithmetic and against the latent's space, and which of the two a step takes."""
import numpy as np
import pytest
import torch

from test_gpu_rasizen import BF16, DEV, mixer_harness, part_close, part_tensors, rand

DIM, ROT, VDIM, WIDTH = 128, 64, 128, 64

pytestmark = pytest.mark.gpu


def layer(heads, rank=512, window=0, scale=0.05, fast=True, **more):
    """(the mixer, its tensors in float64, its runtime)."""
    from sonicboom_amd.parts import Runtime, build_part
    from sonicboom_amd.parts.latent_attention import latent_attention_spec
    from sonicboom_amd.parts.position import rope_interleaved_spec
    spec = latent_attention_spec("a.", WIDTH, heads, DIM, ROT, VDIM, rank, scale, rope_interleaved_spec(ROT, 1e4), window=window, eps=1e-5, **more)
    dev, ref = part_tensors(spec, "bfloat16", scale=0.2)
    rt = Runtime(torch.device(DEV), BF16, fast)
    return build_part(spec, dev, rt), ref, rt


@pytest.mark.parametrize("scale", [-0.05, 0.0, 0.109])
def test_scales_that_stay_in_the_latents_space(scale):
    """Scores times a negative number, all alike, and peaked: the layer's result is the plain kernels'."""
    h = rand(330, WIDTH).to(BF16)
    outs = []
    for fast in (True, False):
        mixer, _, rt = layer(4, scale=scale, fast=fast)
        assert mixer.ukv is None
        outs.append(mixer_harness(mixer, rt)(h, [330], WIDTH))
    part_close(outs[0], outs[1].cpu().numpy(), "bfloat16", f"scale {scale}")


class Fed:
    """A cache for one layer alone: sequences filled with anything, and steps over them."""

    def __init__(self, mixer, rt, tokens, slots=4):
        from sonicboom_amd.cache import PagedCache, group_entries
        self.mixer, self.rt = mixer, rt
        self.cache = PagedCache(group_entries({0: mixer.cache_spec().key()}), tokens, rt.cache_dtype, rt.device, None, max_slots=slots)
        self.rows, v, group = self.cache.entry_views(0)
        from sonicboom_amd.engine.model import LayerBinding
        self.binding = LayerBinding(0, group, self.rows, v, True, None)

    def fill(self, n):
        """A sequence of n cached positions."""
        slot = self.cache.alloc_slot()
        if n:
            self.cache.reserve([slot], [n])
            self.cache.advance([slot], [n])
        return slot

    def step(self, slots, h, n_new, built=None, advance=True):
        """(the layer's output for these rows, whether keys and values were built); built: False keeps them out."""
        from sonicboom_amd.engine.step import StepContext, StepEntry
        self.cache.reserve(slots, n_new)
        ctx = StepContext(self.cache, [StepEntry(s, [0] * n, ()) for s, n in zip(slots, n_new)], self.rt.device, (self.mixer.row_tile,))
        ctx.shared = {self.mixer.built_key: None} if built is False else {}
        x = torch.zeros((sum(n_new), WIDTH), dtype=torch.float32, device=DEV)
        self.mixer.forward(h.to(DEV).contiguous(), x, ctx, self.binding)
        if advance:
            self.cache.advance(slots, n_new)
        else:
            self.cache.trim(slots)
        return x, ctx.shared.get(self.mixer.built_key) is not None


def test_memory_that_does_not_hold_the_built_keys(monkeypatch):
    """Under a limit that the built keys of 120,000 positions (370 MB) do not fit, the step stays in the latent's space."""
    from sonicboom_amd import ops
    monkeypatch.setattr(ops, "latent_built_pays", lambda *a: True)
    mixer, _, rt = layer(4)
    fed = Fed(mixer, rt, 120_064)
    fed.rows.normal_()
    slot, h = fed.fill(119_936), rand(64, WIDTH).to(BF16)
    want, _ = fed.step([slot], h, [64], built=False, advance=False)
    over, built = fed.step([slot], h, [64], advance=False)
    assert built
    part_close(over, want.cpu().numpy(), "bfloat16", "built against the latent's space")
    del over
    torch.cuda.empty_cache()
    most = torch.cuda.memory_reserved() + (200 << 20)
    torch.cuda.set_per_process_memory_fraction(most / torch.cuda.get_device_properties(0).total_memory)
    try:
        got, built = fed.step([slot], h, [64], advance=False)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert not built and torch.equal(got, want)

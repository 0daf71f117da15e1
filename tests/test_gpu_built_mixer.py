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


@pytest.mark.parametrize("scale", [-0.05, 0.0])
def test_a_scale_that_is_not_positive(scale):
    """Scores times a negative number, and all alike: the layer's result is the plain kernels'."""
    h = rand(330, WIDTH).to(BF16)
    outs = []
    for fast in (True, False):
        mixer, _, rt = layer(4, scale=scale, fast=fast)
        outs.append(mixer_harness(mixer, rt)(h, [330], WIDTH))
    part_close(outs[0], outs[1].cpu().numpy(), "bfloat16", f"scale {scale}")

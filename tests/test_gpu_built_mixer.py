"""Latent-attention layers with heads of 128 + 64 numbers and 128 values, whose prompt steps may build keys and values: the layer
against 64-bit arithmetic and against the latent's space, and which of the two a step takes."""
import numpy as np
import pytest
import torch

import test_gpu_fitatar as fitatar
from plain import fitatar_plain as P
from plain import rasizen_plain as R
from test_gpu_rasizen import BF16, DEV, close, config, latent, mixer_harness, part_close, part_tensors, rand, run_cuts

DIM, ROT, VDIM, WIDTH = 128, 64, 128, 64
EPS = 1e-5

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def every_prompt_builds(monkeypatch):
    """Whatever the price says of a step."""
    from sonicboom_amd import ops
    monkeypatch.setattr(ops, "latent_built_pays", lambda *a: True)


def layer(heads, rank=512, window=0, scale=0.05, fast=True, **more):
    """(the mixer, its tensors in float64, its runtime)."""
    from sonicboom_amd.parts import Runtime, build_part
    from sonicboom_amd.parts.latent_attention import latent_attention_spec
    from sonicboom_amd.parts.position import rope_interleaved_spec
    spec = latent_attention_spec("a.", WIDTH, heads, DIM, ROT, VDIM, rank, scale, rope_interleaved_spec(ROT, 1e4), window=window, eps=EPS, **more)
    dev, ref = part_tensors(spec, "bfloat16", scale=0.2)
    rt = Runtime(torch.device(DEV), BF16, fast)
    return build_part(spec, dev, rt), ref, rt


def in_64_bits(ref, h, heads, rank, window, scale):
    mx = {"heads": heads, "dim": DIM, "rot_dim": ROT, "vdim": VDIM, "kv_rank": rank, "scale": scale, "rot": {"base": 1e4, "dims": ROT},
          "mask": {"size": window}}
    hn, at = h.float().numpy(), np.arange(len(h))
    return R.latent_attention_mixer(hn, at, ref, "a.", mx, EPS, R.latent_kv(hn, at, ref, "a.", mx, EPS))


def off(got, want):
    return float(np.linalg.norm(got.double().cpu().numpy() - want) / np.linalg.norm(want))


@pytest.mark.parametrize("heads, rank", [(1, 512), (2, 512), (4, 256), (16, 512)])
@pytest.mark.parametrize("window", [0, 130])
def test_a_layer_whole_and_in_portions(heads, rank, window):
    """A prompt in one step, in two, and in five with single rows between them, whose windows have left pages behind; and how far the
    built form and the latent's space are from 64 bits."""
    mixer, ref, rt = layer(heads, rank, window)
    h = rand(470, WIDTH).to(BF16)
    want = in_64_bits(ref, h, heads, rank, window, 0.05)
    error = {}
    for cuts in ([470], [300, 170], [260, 64, 1, 1, 144]):
        for form in (None, False):
            fed = Fed(mixer, rt, 1024)
            slot, at, outs, built = fed.fill(0), 0, [], []
            for n in cuts:
                out, b = fed.step([slot], h[at:at + n], [n], built=form)
                outs.append(out)
                built.append(b)
                at += n
            if window:
                assert fed.cache.page_table(0, [slot])[0, 0] == -1
            got = torch.cat(outs)
            part_close(got, want, "bfloat16", f"cuts {cuts}, built {built}")
            assert built[0] == (form is None) and not any(b for b, n in zip(built, cuts) if n == 1)
            error[form] = max(error.get(form, 0.0), off(got, want))
    # both round four times on the way (queries or keys, weights, latent results or values, results): the attention alone is between 0.94 and 1.06
    # of the other's error, and all the layer's other roundings are the same
    assert error[None] <= 1.1 * error[False], error


def test_the_price_leads_a_step(monkeypatch):
    """A prompt's rows over few keys go over built keys, few rows behind many do not."""
    from sonicboom_amd import ops
    from sonicboom_amd.ops import kernels
    asked = []
    monkeypatch.setattr(ops, "latent_built_pays", lambda *a: asked.append(a) or kernels.latent_built_pays(*a))
    mixer, _, rt = layer(2)
    fed = Fed(mixer, rt, 20_000)
    fed.rows.normal_(generator=torch.Generator(device=DEV).manual_seed(1))
    assert fed.step([fed.fill(0)], rand(300, WIDTH).to(BF16), [300])[1] and not fed.step([fed.fill(12_000)], rand(3, WIDTH).to(BF16), [3])[1]
    assert [a[:3] for a in asked] == [([300], [0], 0), ([3], [12_000], 0)]


def test_a_step_of_prompts_and_single_rows():
    """A prompt, a sequence that goes on by 40 rows and one by a single row in one step: each has the result that it has alone."""
    heads, rank = 4, 512
    mixer, ref, rt = layer(heads, rank)
    fed = Fed(mixer, rt, 4096)
    rows, before = (300, 40, 1), (0, 77, 200)
    h = [rand(k + n, WIDTH, seed=i).to(BF16) for i, (k, n) in enumerate(zip(before, rows))]
    slots = [fed.fill(0) for _ in rows]
    for s, k, x in zip(slots, before, h):
        if k:
            fed.step([s], x[:k], [k])
    got, built = fed.step(slots, torch.cat([x[k:] for x, k in zip(h, before)]), list(rows))
    assert built
    for part, x, k in zip(got.split(rows), h, before):
        part_close(part, in_64_bits(ref, x, heads, rank, 0, 0.05)[k:], "bfloat16", f"{len(x) - k} rows behind {k}")


def test_queries_of_a_latent_a_gate_a_head_and_a_reader(monkeypatch):
    """Stretched frequencies and a gate a head; and a second layer, with W_uk and W_uv of its own, that reads the first one's rows."""
    from sonicboom_amd import ops
    rank, q_rank, n = 512, 24, 330
    scale = 3.0 / (0.3 * np.sqrt(q_rank * rank * (DIM + ROT)))
    mixer, rt, ref, mx = fitatar.latent_mixer("bfloat16", 4, DIM, ROT, VDIM, rank, q_rank, scale, (4.0, 64, 16.0, 1.0))
    reader, _, ref2, mx2 = fitatar.latent_mixer("bfloat16", 6, DIM, ROT, VDIM, rank, q_rank, scale, (4.0, 64, 16.0, 1.0), seed=50, own=False)
    calls, whole = [], ops.latent_built_attention
    monkeypatch.setattr(ops, "latent_built_attention", lambda *a, **kw: calls.append(a[0].shape[:2]) or whole(*a, **kw))
    h, h2 = rand(n, WIDTH).to(BF16), rand(n, WIDTH, seed=9).to(BF16)
    kept = P.latent_rows(mx, EPS, ref, "a.", h.float().numpy(), np.arange(n))
    part_close(fitatar.mixer_harness(mixer, rt, WIDTH)(h, [n]), P.latent_attention(mx, EPS, ref, "a.", h.float().numpy(), kept), "bfloat16", "own rows")
    both = fitatar.mixer_harness(mixer, rt, WIDTH, reader=reader)
    want = P.latent_attention(mx2, EPS, ref2, "a.", h2.float().numpy(), kept)
    for cuts in ([n], [200, 129, 1]):
        part_close(both(h, cuts, reader_rows=h2), want, "bfloat16", f"a reader, cuts {cuts}")
    assert calls[:3] == [(n, 4), (n, 4), (n, 6)] and calls.count((200, 6)) == 1


def test_a_model_of_two_windows(monkeypatch, tmp_path):
    """Layers without a window and with one, and a reader with another, in one step: whole, in portions and in portions that the engine cuts."""
    import json
    from safetensors.torch import load_file
    from sonicboom_amd import ops
    from sonicboom_amd.engine import DecoderModel, Engine
    from sonicboom_amd.weights import write_random_model
    cfg = config(160, 96, [latent(4, DIM, ROT, VDIM, 256, 0.07, 70, mlp=64), latent(2, DIM, ROT, VDIM, 256, 0.07, 0, kv_from=0),
                           latent(4, DIM, ROT, VDIM, 264, 0.07, 0), latent(4, DIM, ROT, VDIM, 264, 0.07, 150, kv_from=2, mlp=64)], groups=2)
    write_random_model(str(tmp_path), json.loads(json.dumps(cfg)), seed=5, dtype="bfloat16", device=None)
    plain = {k: v.float().numpy().astype(np.float64) for k, v in load_file(str(tmp_path / "model.safetensors")).items()}
    calls, whole = [], ops.latent_built_attention
    monkeypatch.setattr(ops, "latent_built_attention", lambda *a, **kw: calls.append((a[0].shape[0], a[10])) or whole(*a, **kw))
    tokens = [int(t) for t in np.random.default_rng(3).integers(0, 160, size=400)]
    want = R.forward(cfg, plain, tokens)
    model = DecoderModel.from_folder(str(tmp_path), "bfloat16")
    eng = Engine(model, 64 * 20)
    for cuts in ([400], [170, 1, 229]):
        close(run_cuts(eng, tokens, cuts), want, "bfloat16", f"cuts {cuts}")
    assert calls[:4] == [(400, 70), (400, 0), (400, 0), (400, 150)]
    close(run_cuts(Engine(model, 64 * 20, max_step_rows=150), tokens, [400]), want, "bfloat16", "portions")


@pytest.mark.parametrize("scale, rank", [(-0.05, 512), (0.0, 512), (0.109, 512), (0.05, 248)])
def test_layers_that_stay_in_the_latents_space(scale, rank):
    """Scores times a negative number, all alike, and peaked, and latents of few numbers: the layer's result is the plain kernels'."""
    h = rand(330, WIDTH).to(BF16)
    outs = []
    for fast in (True, False):
        mixer, _, rt = layer(4, rank, scale=scale, fast=fast)
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


def test_memory_that_does_not_hold_the_built_keys():
    """Under a limit that the built keys of 120,000 positions (370 MB) do not fit, the step stays in the latent's space."""
    mixer, _, rt = layer(4)
    fed = Fed(mixer, rt, 120_064)
    fed.rows.normal_(generator=torch.Generator(device=DEV).manual_seed(1))
    slot, h = fed.fill(119_936), rand(64, WIDTH).to(BF16)
    want, _ = fed.step([slot], h, [64], built=False, advance=False)
    over, built = fed.step([slot], h, [64], advance=False)
    assert built
    part_close(over, want.cpu().numpy(), "bfloat16", "built against the latent's space")
    del over
    product = mixer.ukv

    def short(*_):
        raise torch.OutOfMemoryError("no room for the product")
    mixer.ukv = short
    got, built = fed.step([slot], h, [64], advance=False)
    assert not built and torch.equal(got, want)
    mixer.ukv = product
    torch.cuda.empty_cache()
    if torch.cuda.memory_reserved() - torch.cuda.memory_allocated() > 100 << 20:
        return                                # (what other tests have left between their tensors would hold them)
    most = torch.cuda.memory_reserved() + (200 << 20)
    torch.cuda.set_per_process_memory_fraction(most / torch.cuda.get_device_properties(0).total_memory)
    try:
        got, built = fed.step([slot], h, [64], advance=False)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert not built and torch.equal(got, want)

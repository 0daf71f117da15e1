"""Prompt steps whose layers are launched by one call give the bits of the same steps launched part by part."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def config(width, heads, kv, inner, vocab=500, layers=3, tied=True):
    return {"architectures": ["Qwen2ForCausalLM"], "num_hidden_layers": layers, "hidden_size": width, "num_attention_heads": heads,
            "num_key_value_heads": kv, "intermediate_size": inner, "vocab_size": vocab, "rope_theta": 10000.0, "rms_norm_eps": 1e-6,
            "max_position_embeddings": 4096, "tie_word_embeddings": tied}


# (sizes whose products go to every kernel; head sizes with tiles of 16, 32 and 64 rows; widths off the stages' 64)
SIZES = [config(128, 2, 2, 320), config(896, 14, 2, 4864), config(256, 4, 1, 712), config(2048, 16, 2, 11008, layers=2), config(160, 10, 2, 96)]
STEPS = [[1, 3], [64], [65], [7, 1, 200, 33], [129], [700, 500], [1536], [1537]]


@pytest.mark.parametrize("cfg", SIZES, ids=lambda c: f"{c['hidden_size']}")
def test_one_call_gives_the_same_bits(cfg, monkeypatch):
    """(Also at the sizes where the launches are the shorter part, which the engine leaves to the parts.)"""
    from sonicboom_amd.engine import DecoderModel, Engine, StepEntry, dense
    monkeypatch.setattr(dense.DenseLayers, "pays", lambda self, rows: True)
    model = DecoderModel.from_random(cfg, 3, "bfloat16", "cuda:0")
    engines = [Engine(model, 64 * 80, max_slots=4) for _ in range(2)]
    engines[1].one_call_layers = False
    rng = np.random.default_rng(5)
    for lengths in STEPS:
        slots = [[e.alloc_slot() for _ in lengths] for e in engines]
        for more in (lengths, [5 for _ in lengths], [1 for _ in lengths]):       # a prompt, a continuation, a token each
            tokens = [rng.integers(0, cfg["vocab_size"], size=n).tolist() for n in more]
            got, want = (e.step([StepEntry(s, t, (0, len(t) - 1)) for s, t in zip(ss, tokens)]) for e, ss in zip(engines, slots))
            assert torch.equal(got, want), (lengths, more)
        for e, ss in zip(engines, slots):
            for s in ss:
                e.free_slot(s)
    from sonicboom_amd.engine.dense import DenseLayers
    assert DenseLayers.of(model, engines[0].bindings) is not None


def same_bits(monkeypatch, cfg, steps, alter=None):
    """Every step of more than single tokens takes one call a layer, whether it pays or not."""
    from sonicboom_amd.engine import DecoderModel, Engine, StepEntry, dense
    monkeypatch.setattr(dense.DenseLayers, "pays", lambda self, rows: True)
    model = DecoderModel.from_random(cfg, 3, "bfloat16", "cuda:0")
    if alter is not None:
        alter(model)
    engines = [Engine(model, 64 * 30, max_slots=4) for _ in range(2)]
    engines[1].one_call_layers = False
    rng = np.random.default_rng(5)
    for lengths in steps:
        tokens = [rng.integers(0, cfg["vocab_size"], size=n).tolist() for n in lengths]
        slots = [[e.alloc_slot() for _ in lengths] for e in engines]
        got, want = (e.step([StepEntry(s, t, (0, len(t) - 1)) for s, t in zip(ss, tokens)]) for e, ss in zip(engines, slots))
        assert torch.equal(got, want), lengths
        for e, ss in zip(engines, slots):
            for s in ss:
                e.free_slot(s)


def test_rows_wider_than_the_pass_that_adds_slices(monkeypatch):
    """The products that join such rows are whole ones, whose own cuts of K need more of the workspace than any slices do."""
    same_bits(monkeypatch, config(14464, 113, 1, 64, layers=1), [[3], [16], [2, 30], [70]])


@pytest.mark.parametrize("cfg", [config(2048, 16, 2, 8192, layers=2), config(3072, 24, 4, 8192, layers=1), config(1024, 8, 2, 4096, layers=2),
                                 config(2048, 16, 4, 5632, layers=1)], ids=lambda c: f"{c['hidden_size']}x{c['intermediate_size']}")
def test_gated_products_that_cut_k_have_the_same_bits(cfg, monkeypatch):
    """Two and three slices of K in the gated product of few rows: the feed-forward's own numbers, before what follows
    rounds them again."""
    from sonicboom_amd import ops
    from sonicboom_amd.engine import DecoderModel, Engine, StepEntry, dense
    monkeypatch.setattr(dense.DenseLayers, "pays", lambda self, rows: True)
    model = DecoderModel.from_random(cfg, 3, "bfloat16", "cuda:0")
    engines = [Engine(model, 64 * 30, max_slots=4) for _ in range(2)]
    engines[1].one_call_layers = False
    mids, run, product = ([], []), ops.DenseStep.run, ops.gemm_bf16

    def watched_run(self, layer, h):
        run(self, layer, h)
        first = self.args.mid - self.args.part               # (`part` stands at the workspace's start)
        mids[0].append(self.kept[-1][first:first + 2 * self.args.n_rows * self.args.inner].clone().view(torch.bfloat16))

    def watched_product(x, w, *args, gated=False, **kw):
        y = product(x, w, *args, gated=gated, **kw)
        if gated:
            mids[1].append(y.clone().reshape(-1))
        return y
    monkeypatch.setattr(ops.DenseStep, "run", watched_run)
    monkeypatch.setattr(ops, "gemm_bf16", watched_product)
    rng = np.random.default_rng(5)
    for lengths in ([2], [3], [2, 6], [9], [16], [40]):
        tokens = [rng.integers(0, cfg["vocab_size"], size=n).tolist() for n in lengths]
        slots = [[e.alloc_slot() for _ in lengths] for e in engines]
        got, want = (e.step([StepEntry(s, t, (0, len(t) - 1)) for s, t in zip(ss, tokens)]) for e, ss in zip(engines, slots))
        assert len(mids[0]) == len(mids[1]) == cfg["num_hidden_layers"]
        for i, (a, b) in enumerate(zip(*mids)):
            assert torch.equal(a, b), (lengths, i)
        assert torch.equal(got, want), lengths
        mids[0].clear(), mids[1].clear()
        for e, ss in zip(engines, slots):
            for s in ss:
                e.free_slot(s)


@pytest.mark.parametrize("other", [(0,), (1,), (2, 3), (1, 3)])
def test_layers_that_differ_stand_between_those_that_do_not(monkeypatch, other):
    """They run part by part, take the norm that the layer before has left and leave the next one's."""
    def alter(model):
        for i in other:
            model.blocks[model.order[i].block].mixer.out_scale = 0.5
    same_bits(monkeypatch, config(128, 2, 2, 320, layers=4), [[2, 3], [65], [7, 1, 200, 33]], alter)


def test_long_steps_take_a_call_a_layer_too(monkeypatch):
    """Sizes at which a call a layer would not pay."""
    same_bits(monkeypatch, SIZES[1], [[700, 500], [1536]])
    same_bits(monkeypatch, SIZES[3], [[129], [300, 41]])


def test_other_models_and_choices_keep_their_parts():
    from sonicboom_amd import ops
    from sonicboom_amd.engine import DecoderModel, Engine, StepEntry
    from sonicboom_amd.engine.dense import DenseLayers
    model = DecoderModel.from_random(SIZES[0], 3, "float32", "cuda:0")
    e = Engine(model, 64 * 4)
    assert DenseLayers.of(model, e.bindings) is None
    model = DecoderModel.from_random(SIZES[0], 3, "bfloat16", "cuda:0")
    e = Engine(model, 64 * 4)
    seen = []
    e.tracer = lambda name, t: seen.append(name)
    s = e.alloc_slot()
    e.step([StepEntry(s, [1, 2, 3], (2,))])
    assert "entry2.after_ffn" in seen
    with ops.gemm_tile_shape(0):
        assert not ops.launchers_choose()
    assert ops.launchers_choose()

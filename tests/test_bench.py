"""The benchmark's kernel table: which products its timers see, what they call them and what they hold them against."""
import torch

import bench
from sonicboom_amd import ops
from sonicboom_amd.parts.linear import Linear


def test_float32_products_are_timed_under_their_matrix(monkeypatch):
    """A projection of float32 weights names its matrix in the way the timers read it (its packed weight is flat)."""
    seen = []
    monkeypatch.setattr(ops, "cast", lambda x, dtype: x)
    monkeypatch.setattr(ops, "gemm_f32", lambda *a, **kw: seen.append(kw.get("packed_shape")))
    for gated in (False, True):
        p = Linear(torch.zeros(6, 5), None, gated=gated)
        p.packed_f32, p.weight = torch.zeros(16 * 16 * (2 if gated else 1)), None
        p(torch.zeros(2, 5), torch.float32)
    assert seen == [(6, 5), (6, 5)]
    assert "gemm_f32" in bench.OpTimer.NAMES
    sizes = {"d": 5, "qw": 4, "kvw": 1, "ff": 9, "v": 100}
    label = bench.OpTimer(sizes)._label
    assert label("gemm_f32", (None, torch.zeros(256)), {"packed_shape": (6, 5)}) == "qkv"
    assert label("gemm_f32", (None, torch.zeros(256)), {"packed_shape": (18, 5), "gated": "silu"}) == "gate_up"


def test_float32_products_are_priced_in_float32():
    cfgs = {"window": 1 << 30, "heads": 16, "rank": 512, "rot": 64, "vocab": 7}
    args = (1.0, 1, 8, 2048, 8, 2048, cfgs)
    n, k, rows = 4096, 2048, 8
    for label, size in (("gemm", 2), ("gemm_f32", 4)):
        share, bound = bench.design_roofline(f"{label} {n}x{k}", *args)
        assert bound == "bytes" and abs(share - (size * (n * k + rows * k) + 4 * rows * n) / (bench.PEAK_HBM_GBS * 1e9) / 1e-6) < 1e-9 * share
    share, bound = bench.design_roofline(f"gemm_f32 {n}x{k}", 1.0, 1, 4096, 4096, 8, 2048, cfgs)
    assert bound == "flops" and abs(share - 2 * 4096 * n * k / bench.VECTOR_F32_FLOPS / 1e-6) < 1e-9 * share

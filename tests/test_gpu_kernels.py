"""Each kernel alone against a plain reference of the same operation, at sizes other
than the engine's tiny configurations: widths that are no power of two, ragged row
counts, head sizes in steps of 16, any number of heads and groups."""
import math

import numpy as np
import pytest
import torch

from plain import qwen2_plain as plain
from plain import sampling_plain
from sonicboom_amd.cache import layout

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
BF16, F32 = torch.bfloat16, torch.float32


def randn(*shape, dtype=F32, scale=1.0, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return (torch.randn(*shape, generator=g) * scale).to(dtype)


def close(got, want, atol, rtol, what=""):
    got = got.detach().float().cpu().double()
    want = torch.as_tensor(want).double()
    assert got.shape == want.shape, f"{what}: {tuple(got.shape)} vs {tuple(want.shape)}"
    assert torch.isfinite(got).all(), f"{what}: not finite"
    err = (got - want).abs()
    bound = atol + rtol * want.abs()
    assert (err <= bound).all(), f"{what}: max |diff| {err.max():.3g} (worst excess {(err - bound).max():.3g})"


# -------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [F32, BF16])
def test_embed(dtype):
    from sonicboom_amd import ops
    table = randn(301, 72, dtype=dtype)
    ids = torch.tensor([0, 300, 7, 7, 150], dtype=torch.int32)
    got = ops.embed(table.to(DEV), ids.to(DEV))
    assert got.dtype == F32 and torch.equal(got.cpu(), table.float()[ids.long()])
    bad = ops.embed(table.to(DEV), torch.tensor([301, -1], dtype=torch.int32, device=DEV))
    assert torch.isnan(bad).all()          # an id outside the table never reads memory it does not own


@pytest.mark.parametrize("n_rows", [7, 300])       # few rows and many rows take different block shapes
@pytest.mark.parametrize("width", [64, 201, 338, 3584, 5000, 8192, 9004])     # up to 4,096, up to 8,192, beyond
@pytest.mark.parametrize("out_dtype, w_dtype", [(F32, F32), (BF16, BF16), (BF16, F32)])
def test_rmsnorm(width, out_dtype, w_dtype, n_rows):
    from sonicboom_amd import ops
    x = randn(n_rows, width, scale=3.0)
    w = (1.0 + randn(width, scale=0.1)).to(w_dtype)
    eps = 1e-5
    want = plain.rms_norm(x.numpy(), w.float().numpy(), eps)
    got = ops.rmsnorm(x.to(DEV), w.to(DEV), eps, out_dtype)
    tol = dict(atol=1e-6, rtol=2e-6) if out_dtype == F32 else dict(atol=1e-2, rtol=8e-3)
    close(got, want, what="rmsnorm", **tol)
    rows = torch.tensor([5, 0, 5], dtype=torch.int32)
    picked = ops.rmsnorm(x.to(DEV), w.to(DEV), eps, out_dtype, rows.to(DEV))
    assert torch.equal(picked.cpu(), got.cpu()[rows.long()])


@pytest.mark.parametrize("width", [64, 100, 3584, 5120, 8192])
@pytest.mark.parametrize("n_slices", [1, 5, 8])
@pytest.mark.parametrize("out_dtype", [F32, BF16])
def test_reduce_resid_norm(width, n_slices, out_dtype):
    """x += slices (+ bias), then the norm of the new x, in one pass: rows narrower and wider than
    what a thread keeps in one group of four."""
    from sonicboom_amd import ops
    rows, eps = 9, 1e-6
    partial = randn(n_slices, rows, width, seed=1)
    x = randn(rows, width, scale=2.0, seed=2)
    bias = randn(width, scale=0.1, seed=3)
    w = 1.0 + randn(width, scale=0.1, seed=4)
    new_x = x.double() + partial.double().sum(0) + bias.double()
    want_y = plain.rms_norm(new_x.float().numpy(), w.numpy(), eps)
    xd = x.to(DEV)
    y = ops.reduce_resid_norm(partial.to(DEV), bias.to(DEV), xd, w.to(DEV), eps, out_dtype)
    close(xd, new_x, atol=2e-6 * n_slices, rtol=2e-6, what="residual")
    tol = dict(atol=2e-5, rtol=2e-5) if out_dtype == F32 else dict(atol=1e-2, rtol=8e-3)
    close(y, want_y, what="normed", **tol)
    # without a norm: only the sum
    xd2 = x.to(DEV)
    assert ops.reduce_resid_norm(partial.to(DEV), None, xd2, None, eps, None) is None
    close(xd2, x.double() + partial.double().sum(0), atol=2e-6 * n_slices, rtol=2e-6, what="sum only")


def test_rmsnorm_reference_vectors():
    """/root/reference/tests/core/test_nn.cpp:172-219."""
    from sonicboom_amd import ops
    x = torch.tensor([[2.0, 2.0, 2.0, 2.0]], device=DEV)
    assert torch.allclose(ops.rmsnorm(x, None, 0.0, F32).cpu(), torch.ones(1, 4), atol=1e-6)
    w3 = torch.full((4,), 3.0, device=DEV)
    assert torch.allclose(ops.rmsnorm(x, w3, 0.0, F32).cpu(), torch.full((1, 4), 3.0), atol=1e-6)
    e = torch.tensor([[1.0, 0.0, 0.0, 0.0]], device=DEV)
    assert torch.equal(ops.rmsnorm(e, None, 0.75, F32).cpu(), torch.tensor([[1.0, 0.0, 0.0, 0.0]]))


def ref_gemm(x, w, bias=None, resid=None):
    y = x.double() @ w.double().T
    if bias is not None:
        y = y + bias.double()
    if resid is not None:
        y = y + resid.double()
    return y


@pytest.mark.parametrize("t, n, k", [(1, 100, 96), (5, 224, 200), (64, 64, 64), (130, 97, 51), (3, 1000, 3584)])
@pytest.mark.parametrize("xd, wd", [(F32, F32), (BF16, BF16), (BF16, F32), (F32, BF16)])
def test_gemm_plain(t, n, k, xd, wd):
    from sonicboom_amd import ops
    x, w = randn(t, k, dtype=xd), randn(n, k, dtype=wd, scale=0.05)
    bias, resid = randn(n, scale=0.1), randn(t, n)
    want = ref_gemm(x, w, bias, resid)
    got = ops.gemm_plain(x.to(DEV), w.to(DEV), bias.to(DEV), resid.to(DEV), F32)
    close(got, want, atol=2e-5 * math.sqrt(k), rtol=1e-5, what="gemm_plain")
    # in place on the residual, and without the extras
    r = resid.to(DEV)
    ops.gemm_plain(x.to(DEV), w.to(DEV), None, r, F32, out=r)
    close(r, ref_gemm(x, w, None, resid), atol=2e-5 * math.sqrt(k), rtol=1e-5, what="gemm_plain in place")


def test_gemm_plain_does_not_depend_on_the_batch():
    """The same row gives the same bits alone and among 200 others."""
    from sonicboom_amd import ops
    x, w = randn(200, 333).to(DEV), randn(150, 333, scale=0.05).to(DEV)
    whole = ops.gemm_plain(x, w, None, None, F32)
    for r in (0, 63, 64, 199):
        alone = ops.gemm_plain(x[r:r + 1].contiguous(), w, None, None, F32)
        assert torch.equal(alone[0], whole[r])


@pytest.mark.parametrize("t, n, k", [(3, 100, 255), (3, 100, 257), (300, 272, 1003), (70, 64, 1022), (2, 48, 4097)])
def test_gemm_f32_of_rows_off_sixteen_bytes(t, n, k):
    """Inner sizes that are no multiple of four, and rows that start between two lines of sixteen bytes: the bits of the plain
    product, plain and gated."""
    from sonicboom_amd import ops
    x, w, bias = randn(t, k).to(DEV), randn(n, k, scale=0.05).to(DEV), randn(n).to(DEV)
    off = torch.empty(t * k + 1, device=DEV)[1:].view(t, k).copy_(x)
    want, both = ops.gemm_plain(x, w, bias, None, F32), ops.gemm_plain(x, w, None, None, F32)
    for rows in (x, off):
        assert torch.equal(ops.gemm_f32(rows, ops.pack_weight_f32(w), bias, None, F32, (n, k)), want)
        assert torch.equal(ops.gemm_f32(rows, ops.pack_weight_f32(w, True), None, None, F32, (n, k), gated="silu"), ops.silu_mul(both, F32))


@pytest.mark.parametrize("t, n, k", [(2100, 520, 1100), (1030, 1100, 2060), (2048, 768, 64), (3, 33000, 2050)])
@pytest.mark.parametrize("xd, wd", [(F32, F32), (BF16, BF16), (BF16, F32), (F32, BF16)])
def test_gemm_plain_many_rows_give_the_bits_of_one(t, n, k, xd, wd):
    """The form for many tiles and the form for few: the same bits of every element, over several segments of K."""
    from sonicboom_amd import ops
    x, w, bias, resid = randn(t, k).to(xd).to(DEV), randn(n, k, scale=0.05).to(wd).to(DEV), randn(n).to(DEV), randn(t, n).to(DEV)
    whole = ops.gemm_plain(x, w, bias, resid, F32)
    rows = [0, 1, t // 2, t - 1]
    close(whole[rows], ref_gemm(x[rows].cpu(), w.cpu(), bias.cpu(), resid[rows].cpu()), atol=2e-5 * math.sqrt(k), rtol=1e-5)
    for cols in (slice(0, 200), slice(n - 100, n)):
        few = ops.gemm_plain(x[rows], w[cols].contiguous(), bias[cols].contiguous(), resid[rows][:, cols].contiguous(), F32)
        assert torch.equal(whole[rows][:, cols], few)


@pytest.mark.parametrize("t, n, k", [(1, 16, 16), (3, 70, 33), (16, 33, 1020), (17, 300, 1024), (33, 130, 1025), (64, 257, 2052),
                                     (65, 64, 4864), (2, 12300, 48), (700, 272, 9000)])
def test_gemm_f32_packed_gives_the_bits_of_the_plain_product(t, n, k):
    """Tile edges, remainders of 4, 16 and 1,024 k, every tile shape of the launcher, rows off 16 bytes."""
    from sonicboom_amd import ops
    x, w = randn(t, k).to(DEV), randn(n, k, scale=0.05).to(DEV)
    bias, resid = randn(n, scale=0.1).to(DEV), randn(t, n).to(DEV)
    want = ops.gemm_plain(x, w, bias, resid, F32)
    # the sum of a row of k products, each side within k half-ulps of its chains
    close(want, ref_gemm(x.cpu(), w.cpu(), bias.cpu(), resid.cpu()), atol=2e-5 * math.sqrt(k), rtol=1e-5, what="gemm_plain")
    packed = ops.pack_weight_f32(w)
    assert torch.equal(ops.gemm_f32(x, packed, bias, resid, F32, (n, k)), want)
    assert torch.equal(ops.gemm_f32(x[t - 1:], packed, bias, resid[t - 1:].contiguous(), F32, (n, k)), want[t - 1:])
    off = torch.empty(t * k + 1, device=DEV)[1:].view(t, k).copy_(x)
    assert torch.equal(ops.gemm_f32(off, packed, bias, resid, F32, (n, k)), want)
    if n % 2 == 0:
        both = ops.gemm_plain(x, w, None, None, F32)
        gated = ops.gemm_f32(x, ops.pack_weight_f32(w, True), None, None, F32, (n, k), gated="silu")
        assert torch.equal(gated, ops.silu_mul(both, F32))


@pytest.mark.parametrize("t, n, k", [(18, 4880, 64), (64, 2100, 896), (200, 1216, 896), (520, 1152, 900), (1100, 272, 512), (1100, 1152, 896)])
def test_gemm_f32_every_tile_of_one_segment_gives_the_same_bits(t, n, k):
    """One segment of K: sizes on either side of what chooses among the tiles for more than sixteen rows, plain and gated."""
    from sonicboom_amd import ops
    x, w = randn(t, k).to(DEV), randn(n, k, scale=0.05).to(DEV)
    want = ops.gemm_plain(x, w, None, None, F32)
    assert torch.equal(ops.gemm_f32(x, ops.pack_weight_f32(w), None, None, F32, (n, k)), want)
    gated = ops.gemm_f32(x, ops.pack_weight_f32(w, True), None, None, F32, (n, k), gated="silu")
    assert torch.equal(gated, ops.silu_mul(want, F32))


@pytest.mark.parametrize("t", [1, 3, 16])
@pytest.mark.parametrize("n, k", [(896, 4864), (33, 1028), (300, 2048), (17, 8192)])
def test_gemm_f32_segments_add_up_to_the_same_bits(t, n, k):
    """The planes of K's segments, added in order, and through the pass that adds them to a residual and norms."""
    from sonicboom_amd import ops
    from sonicboom_amd.parts.linear import Linear
    x, w, resid = randn(t, k).to(DEV), randn(n, k, scale=0.05).to(DEV), randn(t, n).to(DEV)
    packed = ops.pack_weight_f32(w)
    part = ops.gemm_f32_partial(x, packed, (n, k))
    total = part[0].clone()
    for plane in part[1:]:
        total = total + plane
    assert torch.equal(total, ops.gemm_f32(x, packed, None, None, F32, (n, k)))
    want = ops.gemm_f32(x, packed, None, resid, F32, (n, k))
    got = resid.clone()
    Linear(w, None, fast=True).add_into(x, got)
    assert torch.equal(got, want)
    if n % 4 == 0:
        assert torch.equal(ops.reduce_resid_norm(part, None, resid, torch.ones(n, device=DEV), 1e-6, F32),
                           ops.rmsnorm(want, torch.ones(n, device=DEV), 1e-6, F32))
    for rows, inner in ((17, k), (t, 1024), (t, 8196), (t, 1030)):     # more rows, one segment, nine, no whole fours
        assert ops.gemm_f32_partial(torch.zeros(rows, inner, device=DEV), torch.zeros((n + 15) // 16 * 16 * ((inner + 15) // 16 * 16), device=DEV),
                                    (n, inner)) is None


@pytest.mark.parametrize("t", [1, 5, 16, 17, 33, 64, 65, 128, 300])
@pytest.mark.parametrize("n, k", [(96, 64), (100, 96), (224, 200), (3584, 512), (1000, 3584), (72, 18944 // 8)])
def test_gemm_bf16_matrix_cores(t, n, k):
    from sonicboom_amd import ops
    x, w = randn(t, k, dtype=BF16), randn(n, k, dtype=BF16, scale=0.05)
    bias, resid = randn(n, scale=0.1), randn(t, n)
    want = ref_gemm(x, w, bias, resid)
    got = ops.gemm_bf16(x.to(DEV), w.to(DEV), bias.to(DEV), resid.to(DEV), F32)
    assert got is not None
    close(got, want, atol=3e-5 * math.sqrt(k), rtol=1e-5, what=f"gemm_bf16 t={t}")
    got16 = ops.gemm_bf16(x.to(DEV), w.to(DEV), None, None, BF16)
    close(got16, ref_gemm(x, w), atol=2e-2, rtol=8e-3, what=f"gemm_bf16 bf16 out t={t}")
    r = resid.to(DEV)
    ops.gemm_bf16(x.to(DEV), w.to(DEV), None, r, F32, out=r)
    close(r, ref_gemm(x, w, None, resid), atol=3e-5 * math.sqrt(k), rtol=1e-5, what="in place")


@pytest.mark.parametrize("t", [1, 8, 40, 64, 65, 200])
@pytest.mark.parametrize("inner, k", [(100, 96), (224, 200), (18944 // 4, 512)])
def test_gemm_bf16_gated(t, inner, k):
    from sonicboom_amd import ops
    x, w = randn(t, k, dtype=BF16), randn(2 * inner, k, dtype=BF16, scale=0.1)
    gu = x.double() @ w.double().T
    g, u = gu[:, :inner], gu[:, inner:]
    want = g / (1.0 + torch.exp(-g)) * u
    got = ops.gemm_bf16(x.to(DEV), w.to(DEV), None, None, F32, gated=True)
    close(got, want, atol=1e-4 * math.sqrt(k), rtol=1e-4, what=f"gated t={t}")


def gelu_tanh(g):
    """0.5 g (1 + tanh(sqrt(2/pi) g (1 + 0.044715 g^2))), /root/reference/core/src/nn/activation.cpp:27-36."""
    return 0.5 * g * (1.0 + torch.tanh(0.7978845608028654 * g * (1.0 + 0.044715 * g * g)))


@pytest.mark.parametrize("t", [1, 8, 40, 64, 65, 128, 300])
def test_gemm_bf16_gate_activations(t):
    """The gate's activation is an argument of every product kernel and of the elementwise
    kernel: SiLU, the tanh form of GELU and max(g, 0), through the stream, the K-splitting and the
    tiled kernels, against the formula and against torch's own GELU."""
    from sonicboom_amd import ops
    inner, k = 1040, 264
    x, w = randn(t, k, dtype=BF16), randn(2 * inner, k, dtype=BF16, scale=0.15)
    gu = x.double() @ w.double().T
    g, u = gu[:, :inner], gu[:, inner:]
    assert torch.allclose(gelu_tanh(g), torch.nn.functional.gelu(g, approximate="tanh"), atol=1e-12)
    want = {"silu": g / (1.0 + torch.exp(-g)) * u, "gelu_tanh": gelu_tanh(g) * u, "relu": torch.clamp(g, min=0.0) * u}
    assert (want["silu"] - want["gelu_tanh"]).abs().max() > 0.05          # the two differ visibly
    packed = ops.pack_weight(w.to(DEV), True)
    assert (want["relu"] - want["gelu_tanh"]).abs().max() > 0.05
    for act in ("silu", "gelu_tanh", "relu"):
        for which in ("stream", "skinny", "tiled"):
            if (which == "stream" and t > 128) or (which == "skinny" and t > 64):
                continue
            with ops.gemm_few_rows_kernel(which):
                got = ops.gemm_bf16(x.to(DEV), packed, None, None, F32, gated=act, packed_shape=(2 * inner, k))
            close(got, want[act], atol=1e-4 * math.sqrt(k), rtol=1e-4, what=f"{act} through {which}, t={t}")
        got = ops.gate_mul(gu.float().to(DEV), F32, act)
        close(got, want[act], atol=1e-5, rtol=1e-5, what=f"{act}, elementwise")
    with pytest.raises(ops.KernelLibraryError, match="unknown gate activation"):
        ops.gate_mul(gu.float().to(DEV), F32, "softsign")


@pytest.mark.parametrize("shape", [0, 1, 2])
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("t, n, k", [(65, 100, 96), (300, 224, 200), (520, 264, 128), (257, 1000, 448), (130, 72, 2368)])
def test_gemm_bf16_every_tile_shape(shape, packed, t, n, k):
    """Each tile shape of the tiled product, with K a multiple of the stage or not, rows and
    columns that end inside a tile, plain and packed weights, plain and gated."""
    from sonicboom_amd import ops
    x, w = randn(t, k, dtype=BF16), randn(n, k, dtype=BF16, scale=0.05)
    bias, resid = randn(n, scale=0.1), randn(t, n)
    wd = w.to(DEV)
    # plain (unpacked) weights always take the 128 x 128 tile
    with ops.gemm_tile_shape(shape):
        got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(wd) if packed else wd, bias.to(DEV), resid.to(DEV), F32,
                            packed_shape=(n, k) if packed else None)
        close(got, ref_gemm(x, w, bias, resid), atol=3e-5 * math.sqrt(k), rtol=1e-5, what=f"shape {shape}")
        inner = n // 2
        gu = x.double() @ w[:2 * inner].double().T
        g, u = gu[:, :inner], gu[:, inner:]
        wg = wd[:2 * inner].contiguous()
        got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(wg, True) if packed else wg, None, None, F32, gated=True,
                            packed_shape=(2 * inner, k) if packed else None)
        close(got, g / (1.0 + torch.exp(-g)) * u, atol=1e-4 * math.sqrt(k), rtol=1e-4, what=f"gated shape {shape}")


@pytest.mark.parametrize("shape, path", [(0, "direct"), (1, "direct"), (2, "direct"), (3, "direct"), (4, "direct"),
                                         (2, "direct, a block a tile"), (0, "registers"), (2, "registers")])
@pytest.mark.parametrize("t, n, k", [(65, 100, 64), (300, 226, 192), (520, 264, 128), (257, 1001, 448), (130, 72, 2368)])
def test_gemm_bf16_every_path(shape, path, t, n, k):
    """The kernel that loads its tiles straight into LDS (inner sizes in 64s, packed weights) and
    the one that stages them through registers, forced for every tile shape: rows and columns
    that end inside a tile, widths that are no multiple of 4 (single stores in the epilogue),
    bias and residual, bfloat16 and float32 results, plain and gated."""
    from sonicboom_amd import ops
    x, w = randn(t, k, dtype=BF16), randn(n, k, dtype=BF16, scale=0.05)
    bias, resid = randn(n, scale=0.1), randn(t, n)
    wd = w.to(DEV)
    with ops.gemm_tile_shape(shape, path):
        got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(wd), bias.to(DEV), resid.to(DEV), F32, packed_shape=(n, k))
        close(got, ref_gemm(x, w, bias, resid), atol=3e-5 * math.sqrt(k), rtol=1e-5, what=f"shape {shape} {path}")
        got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(wd), bias.to(DEV), None, BF16, packed_shape=(n, k))
        close(got, ref_gemm(x, w, bias, None), atol=0.01 * math.sqrt(k) * 0.05 + 0.01, rtol=0.01, what=f"bf16 shape {shape} {path}")
        inner = n // 2
        gu = x.double() @ w[:2 * inner].double().T
        g, u = gu[:, :inner], gu[:, inner:]
        wg = wd[:2 * inner].contiguous()
        for act, want in (("silu", g / (1.0 + torch.exp(-g)) * u),
                          ("gelu_tanh", 0.5 * g * (1 + torch.tanh(0.7978845608028654 * g * (1 + 0.044715 * g * g))) * u)):
            got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(wg, True), None, None, F32, gated=act, packed_shape=(2 * inner, k))
            close(got, want, atol=1e-4 * math.sqrt(k), rtol=1e-4, what=f"gated {act} shape {shape} {path}")


@pytest.mark.parametrize("t, n, k", [(65, 100, 64), (183, 226, 192), (288, 264, 128), (300, 1001, 448), (65, 72, 2368)])
@pytest.mark.parametrize("big", [False, True])
def test_gemm_bf16_tiles_of_64_rows(t, n, k, big):
    """Straight into LDS in one round over the CUs (four stages in flight) and in more (two): rows, columns and
    stage counts that end inside a tile or a round of the buffers."""
    from sonicboom_amd import ops
    t, n = (t * 9, n * 9) if big else (t, n)
    x, w = randn(t, k, dtype=BF16), randn(n, k, dtype=BF16, scale=0.05)
    wd, inner = w.to(DEV), n // 2
    want = ref_gemm(x, w, None, None)
    for shape in (5, 0):
        with ops.gemm_tile_shape(shape, "direct"):
            got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(wd), None, None, F32, packed_shape=(n, k))
            close(got, want, atol=3e-5 * math.sqrt(k), rtol=1e-5, what=f"shape {shape}")
            g, u = want[:, :inner].double(), want[:, inner:2 * inner].double()
            got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(wd[:2 * inner].contiguous(), True), None, None, F32,
                                gated=True, packed_shape=(2 * inner, k))
            close(got, g / (1.0 + torch.exp(-g)) * u, atol=1e-4 * math.sqrt(k), rtol=1e-4, what=f"gated shape {shape}")


@pytest.mark.parametrize("t, n, k", [(65, 896, 896), (183, 1536, 8960), (288, 900, 4864), (183, 3584, 1280), (512, 1100, 640),
                                     (1500, 3584, 4096), (100, 64, 192)])
def test_gemm_bf16_k_slices_of_tiled_products(t, n, k):
    """The raw product in K slices, at sizes that take each of its tiles."""
    from sonicboom_amd import ops
    x, w = randn(t, k, dtype=BF16), randn(n, k, dtype=BF16, scale=0.05)
    part = ops.gemm_bf16_partial(x.to(DEV), ops.pack_weight(w.to(DEV)), packed_shape=(n, k))
    got = part.sum(0) if part is not None else ops.gemm_bf16(x.to(DEV), ops.pack_weight(w.to(DEV)), None, None, F32, packed_shape=(n, k))
    close(got, ref_gemm(x, w, None, None), atol=3e-5 * math.sqrt(k), rtol=1e-5, what="slices")


def test_k_slices_of_prompts_of_some_hundred_rows():
    """How a prompt's product is cut over K: in fewer slices as rows grow, and whole where slices cost more to write and read than they save."""
    from sonicboom_amd import ops
    slices = ops.library.core().sb_gemm_mfma_slices
    assert [slices(t, 896, 896, 1) for t in (183, 400, 1200)] == [3, 2, 1]
    assert [slices(t, 4096, 14336, 1) for t in (183, 288, 400)] == [4, 2, 2] and slices(640, 1536, 8960, 1) == 4


def test_silu_of_the_tiled_product_over_its_range():
    """A product that hands the gate its numbers as they are, over the float32 range: against 64-bit arithmetic to
    two units of the last of 24 bits, and where e^-g runs out of the range to what is as good as zero."""
    from sonicboom_amd import ops
    g = torch.cat([torch.linspace(-120, 120, 4001), torch.logspace(-30, 38, 400), -torch.logspace(-30, 38, 400),
                   torch.zeros(1)]).to(BF16)
    x = torch.zeros(g.numel(), 32, dtype=BF16)
    x[:, 0] = g
    x[:, 1] = 1.0
    w = torch.zeros(2, 32, dtype=BF16)
    w[0, 0] = 1.0
    w[1, 1] = 1.0
    got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(w.to(DEV), True), None, None, F32, gated=True, packed_shape=(2, 32)).cpu()[:, 0].double()
    z = x[:, 0].double()
    want = z / (1.0 + torch.exp(-z))
    ok = z > -80.0
    assert ((got - want).abs()[ok] <= 2.5e-7 * want.abs()[ok]).all()
    assert (got[~ok].abs() <= 1e-30).all()


@pytest.mark.parametrize("shape, path", [(None, None), (0, "registers"), (2, "registers"), (0, "direct"), (2, "direct")])
def test_silu_of_the_tiled_product_keeps_float32(shape, path):
    """Every kernel's epilogue, over all numbers whose e^-g lies in the float32 range: within two units of the last of 24
    bits (one of the exponential, a half each of the sum and the quotient); past it the values of the full division."""
    from sonicboom_amd import ops
    g = torch.cat([torch.linspace(-88.7, 120.0, 20001), torch.logspace(-30, 38, 500), -torch.logspace(-30, 1.9, 500),
                   torch.tensor([0.0, -88.8, -89.0, -1e3, -3e38, math.inf, -math.inf, math.nan, 1.0, 86.99, 87.0, -86.99, -87.0])])
    x = torch.zeros(g.numel(), 64, dtype=BF16)
    rest = g.clone()
    for i in range(3):                           # three bfloat16 parts add up to the float32 number exactly
        x[:, i] = torch.where(torch.isinf(g), torch.zeros_like(rest), rest).to(BF16)
        rest = rest - x[:, i].float()
    x[:, 3] = 1.0
    x[:, 4] = torch.where(torch.isinf(g), torch.sign(g) * 1e10, torch.zeros_like(g)).to(BF16)    # an infinite product of finite numbers
    w = torch.zeros(2, 64, dtype=BF16)
    w[0, :3] = 1.0
    w[0, 4] = 1e38
    w[1, 3] = 1.0
    with ops.gemm_tile_shape(shape, path):
        got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(w.to(DEV), True), None, None, F32, gated=True, packed_shape=(2, 64))
    got = got.cpu()[:, 0].double()
    finite = torch.isfinite(g)
    z = torch.where(finite, x[:, :3].double().sum(1), torch.zeros(()).double())
    assert ((z - g.double()).abs()[finite] <= 2.0 ** -23 * g.double().abs()[finite]).all()
    want = z / (1.0 + torch.exp(-z))
    ok = finite & (z >= -88.71)
    assert ((got - want).abs()[ok] <= 2.5e-7 * want.abs()[ok]).all()
    assert (got.abs()[finite & ~ok] <= 3e-37).all()
    assert got[g == math.inf].item() == math.inf and torch.isnan(got[g.isnan() | (g == -math.inf)]).all()


def test_gemm_bf16_blocks_that_go_from_tile_to_tile():
    """More 256 x 256 tiles than the GPU has CUs: the blocks of the kernel that loads straight into
    LDS go on to a second tile, whose first stage the first tile's last stage has loaded; in
    bands of eight tiles along the rows, the last band lower.  Every tile has a value of its own."""
    from sonicboom_amd import ops
    t, n, k = 4400, 4200, 128                  # 18 x 17 = 306 tiles; gated: 18 x 33 tiles of 256 x 128
    x, w = randn(t, k, dtype=BF16), randn(n, k, dtype=BF16, scale=0.05)
    want = ref_gemm(x, w, None, None)
    wd = w.to(DEV)
    # (tiles of 192 rows: 23 x 17 = 391)
    for shape, path in ((2, "direct"), (2, "direct, a block a tile"), (4, "direct")):
        with ops.gemm_tile_shape(shape, path):
            got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(wd), None, None, F32, packed_shape=(n, k))
            close(got, want, atol=3e-5 * math.sqrt(k), rtol=1e-5, what=f"{shape} {path}")
            inner = n // 2
            g, u = want[:, :inner].double(), want[:, inner:2 * inner].double()
            got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(wd[:2 * inner].contiguous(), True), None, None, F32,
                                gated=True, packed_shape=(2 * inner, k))
            close(got, g / (1.0 + torch.exp(-g)) * u, atol=1e-4 * math.sqrt(k), rtol=1e-4, what=f"gated {shape} {path}")


@pytest.mark.parametrize("shape", [1, 2])
@pytest.mark.parametrize("t, n, k", [(300, 520, 1024), (300, 520, 16448), (1000, 1800, 8192), (4400, 4200, 128), (4400, 4200, 192), (4400, 4200, 256),
                                     (4400, 4200, 320), (4400, 4200, 1088), (4400, 4200, 8128), (4400, 4200, 8192)])
def test_gemm_bf16_blocks_that_go_on_give_the_bits_of_a_block_a_tile(shape, t, n, k):
    """Tiles of 256 x 128 and 256 x 256: blocks that go on to a second tile, whose first stages are loaded in the last ones of
    the first (4,400 x 4,200: 594 and 306 tiles on 256 CUs), against a block for every tile, from the least inner size that
    goes on; and few tiles, where no block does."""
    from sonicboom_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(3)
    x = torch.randn(t, k, generator=gen, device=DEV).to(BF16)
    w = ops.pack_weight((torch.randn(n, k, generator=gen, device=DEV) * 0.05).to(BF16))
    resid = torch.randn(t, n, generator=gen, device=DEV)
    got = {}
    for path in ("direct", "direct, a block a tile"):
        with ops.gemm_tile_shape(shape, path):
            got[path] = ops.gemm_bf16(x, w, None, resid, F32, packed_shape=(n, k))
    assert torch.equal(*got.values())
    with ops.gemm_tile_shape(0, "registers"):
        other = ops.gemm_bf16(x, w, None, resid, F32, packed_shape=(n, k))
    # (the sums in another order: k terms of size 0.05, 2^-24 each of sums of size sqrt(k) 0.05)
    assert (got["direct"] - other).abs().max().item() <= 3e-5 * math.sqrt(k)


@pytest.mark.parametrize("k", [64, 128, 192, 256, 320, 384, 448, 512, 1088])
@pytest.mark.parametrize("t, n", [(1, 5), (257, 300), (4400, 4200)])
def test_gemm_bf16_largest_tiles_of_every_few_stages(t, n, k):
    """256 x 256 tiles of one to eight 64s of k: shorter and longer than the rings of buffers that the loads run ahead in,
    every position of the rings at a tile's end, in one tile, a few, and blocks that go on to a second one; gated too."""
    from sonicboom_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(k)
    x = torch.randn(t, k, generator=gen, device=DEV).to(BF16)
    w = (torch.randn(n // 2 * 2, k, generator=gen, device=DEV) * 0.05).to(BF16)
    want = x.double() @ w.double().T
    for path in ("direct", "direct, a block a tile"):
        with ops.gemm_tile_shape(2, path):
            got = ops.gemm_bf16(x, ops.pack_weight(w), None, None, F32, packed_shape=tuple(w.shape))
            # k terms of size 0.05, 2^-24 each of sums of size sqrt(k) 0.05
            assert (got - want).abs().max().item() <= 3e-5 * math.sqrt(k), path
            got = ops.gemm_bf16(x, ops.pack_weight(w, True), None, None, F32, gated=True, packed_shape=tuple(w.shape))
            g, u = want.chunk(2, dim=1)
            assert (got - g * torch.sigmoid(g) * u).abs().max().item() <= 1e-4 * math.sqrt(k), path


@pytest.mark.parametrize("k", [64, 128, 192, 256, 448, 1088])
@pytest.mark.parametrize("t, n", [(1, 5), (257, 300), (4400, 2200)])
def test_gemm_bf16_tall_tiles_of_every_few_stages(t, n, k):
    """256 x 128 tiles straight into LDS, likewise; with a bias and a residual in place."""
    from sonicboom_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(k)
    x = torch.randn(t, k, generator=gen, device=DEV).to(BF16)
    w = (torch.randn(n // 2 * 2, k, generator=gen, device=DEV) * 0.05).to(BF16)
    bias, resid = torch.randn(n // 2 * 2, generator=gen, device=DEV), torch.randn(t, n // 2 * 2, generator=gen, device=DEV)
    want = x.double() @ w.double().T
    for path in ("direct", "direct, a block a tile"):
        with ops.gemm_tile_shape(1, path):
            got = resid.clone()
            ops.gemm_bf16(x, ops.pack_weight(w), bias, got, F32, out=got, packed_shape=tuple(w.shape))
            # k terms of size 0.05, 2^-24 each of sums of size sqrt(k) 0.05
            assert (got - (want + bias.double() + resid.double())).abs().max().item() <= 3e-5 * math.sqrt(k), path
            got = ops.gemm_bf16(x, ops.pack_weight(w, True), None, None, F32, gated=True, packed_shape=tuple(w.shape))
            g, u = want.chunk(2, dim=1)
            assert (got - g * torch.sigmoid(g) * u).abs().max().item() <= 1e-4 * math.sqrt(k), path


def test_gemm_bf16_direct_path_refuses_what_it_cannot_take():
    from sonicboom_amd import ops
    x, w = randn(70, 96, dtype=BF16).to(DEV), randn(64, 96, dtype=BF16).to(DEV)
    with ops.gemm_tile_shape(0, "direct"):
        with pytest.raises(ops.KernelLibraryError, match="inner size in 64s"):
            ops.gemm_bf16(x, ops.pack_weight(w), None, None, F32, packed_shape=(64, 96))
    with ops.gemm_tile_shape(3, "registers"):
        with pytest.raises(ops.KernelLibraryError, match="direct path only"):
            ops.gemm_bf16(x, ops.pack_weight(w), None, None, F32, packed_shape=(64, 96))


@pytest.mark.parametrize("t", [1, 3, 8, 9])
@pytest.mark.parametrize("n, k", [(16, 32), (33, 264), (352, 2048), (1000, 520)])
@pytest.mark.parametrize("gate", ["silu", "gelu_tanh"])
def test_gemm_bf16_gated_few_rows_of_small_matrices(t, n, k, gate):
    """The kernel whose waves split K inside a block, for rows without an unfinished norm (up to eight), and the one past it."""
    from sonicboom_amd import ops
    x, w = randn(t, k, dtype=BF16), randn(2 * n, k, dtype=BF16, scale=0.05)
    got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(w.to(DEV), True), None, None, BF16, gated=gate, packed_shape=(2 * n, k))
    g, u = ref_gemm(x, w, None, None).double().chunk(2, dim=1)
    act = g / (1.0 + torch.exp(-g)) if gate == "silu" else torch.nn.functional.gelu(g, approximate="tanh")
    close(got, act * u, atol=1e-4 * math.sqrt(k), rtol=8e-3, what=gate)      # one rounding to bfloat16


@pytest.mark.parametrize("t", [1, 3, 8])
@pytest.mark.parametrize("n, k", [(5, 8), (33, 264), (100, 1032), (352, 1544), (200, 2048), (100, 2600), (77, 3080), (48, 3592), (130, 4096),
                                  (5632, 2048), (8192, 1024), (64, 4104), (3056, 4104), (3057, 4104), (3070, 8192),
                                  (3070, 8200)])
def test_gemm_bf16_gated_few_rows_have_the_bits_of_more(t, n, k):
    """Up to eight rows take one launch whose blocks keep the slices of K to themselves, nine go through scratch and a second
    kernel: one to eight slices, chains of unequal length and none, matrices on either side of the counts that cut K further."""
    from sonicboom_amd import ops
    x, w = randn(9, k, dtype=BF16).to(DEV), randn(2 * n, k, dtype=BF16, scale=0.05).to(DEV)
    packed = ops.pack_weight(w, True)
    for gate in ("silu", "gelu_tanh", "relu"):
        for dtype in (BF16, F32):
            with ops.gemm_few_rows_kernel("skinny"):
                want = ops.gemm_bf16(x, packed, None, None, dtype, gated=gate, packed_shape=(2 * n, k))
                got = ops.gemm_bf16(x[:t].clone(), packed, None, None, dtype, gated=gate, packed_shape=(2 * n, k))
                rows = ops.gemm_bf16(x[:t].clone(), w, None, None, dtype, gated=gate)
            assert torch.equal(got, want[:t]), (gate, dtype)
            assert torch.equal(rows, want[:t]), (gate, dtype)
            assert torch.equal(ops.gemm_bf16(x[:t].clone(), packed, None, None, dtype, gated=gate, packed_shape=(2 * n, k)), got)


@pytest.mark.parametrize("waves", [0, 3])
@pytest.mark.parametrize("t, n, k", [(1, 16, 32), (17, 100, 96), (40, 1000, 520), (65, 264, 2368), (128, 33, 264)])
def test_gemm_bf16_stream_kernel_of_few_waves(t, waves, n, k):
    """Three waves a block, which matrices of few tiles take: every count of row tiles, columns that end inside a
    tile and inside a block, K inside a staged chunk; plain and gated."""
    from sonicboom_amd import ops
    x, w = randn(t, k, dtype=BF16), randn(2 * n, k, dtype=BF16, scale=0.05)
    resid, wd = randn(t, n), w.to(DEV)
    with ops.gemm_few_rows_kernel("stream", waves):
        got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(wd[:n].contiguous()), None, resid.to(DEV), F32, packed_shape=(n, k))
        gated = ops.gemm_bf16(x.to(DEV), ops.pack_weight(wd, True), None, None, F32, gated=True, packed_shape=(2 * n, k))
    close(got, ref_gemm(x, w[:n], None, resid), atol=3e-5 * math.sqrt(k), rtol=1e-5, what="plain")
    g, u = ref_gemm(x, w, None, None).double().chunk(2, dim=1)
    close(gated, g / (1.0 + torch.exp(-g)) * u, atol=1e-4 * math.sqrt(k), rtol=1e-4, what="gated")


@pytest.mark.parametrize("t", [1, 16, 17, 40, 64, 65, 100, 128])
@pytest.mark.parametrize("waves", [0, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("n, k", [(100, 96), (1000, 520), (264, 2368), (4099, 264)])
def test_gemm_bf16_stream_kernel(t, waves, n, k):
    """The kernel for few rows against wide matrices, at every count of waves per block: K
    shorter than one staged chunk, ending inside a chunk and inside a k-step; columns that end
    inside a tile and inside a block; plain with bias and residual, and gated."""
    from sonicboom_amd import ops
    x, w = randn(t, k, dtype=BF16), randn(n, k, dtype=BF16, scale=0.05)
    bias, resid = randn(n, scale=0.1), randn(t, n)
    wd = w.to(DEV)
    with ops.gemm_few_rows_kernel("stream", waves):
        got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(wd), bias.to(DEV), resid.to(DEV), F32, packed_shape=(n, k))
        close(got, ref_gemm(x, w, bias, resid), atol=3e-5 * math.sqrt(k), rtol=1e-5, what="stream")
        got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(wd), None, None, BF16, packed_shape=(n, k))
        close(got.float(), ref_gemm(x, w), atol=2e-2, rtol=1e-2, what="stream, bfloat16 out")
        inner = n // 2
        wg = wd[:2 * inner].contiguous()
        gu = x.double() @ w[:2 * inner].double().T
        g, u = gu[:, :inner], gu[:, inner:]
        got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(wg, True), None, None, F32, gated=True,
                            packed_shape=(2 * inner, k))
        close(got, g / (1.0 + torch.exp(-g)) * u, atol=1e-4 * math.sqrt(k), rtol=1e-4, what="stream, gated")


@pytest.mark.parametrize("t", [8, 17, 64, 100])
def test_gemm_bf16_wide_matrix_with_few_rows(t):
    """Up to 128 rows against a packed matrix wide enough for the stream kernel, and one wave's
    worth of columns less (which stays with the kernel that splits K), plain and gated: the
    choice between the kernels changes no result."""
    from sonicboom_amd import ops
    from sonicboom_amd.ops import kernels
    k = 64
    x = randn(t, k, dtype=BF16)
    edge = 4 * kernels.STREAM_MIN_BLOCKS
    # (the library's choice does change there: 0 the stream kernel, 1 the one that splits K; both leave 65 rows and more of such sizes to the tiled one)
    for gate, per in ((0, 32), (1, 16)):
        took = [ops.library.core().sb_gemm_bf16_kernel(t, n, gate, 1) for n in (edge * per, edge * per - per)]
        assert took == ([0, 1] if t <= 64 else [2, 2])
    for n in (edge * 32, edge * 32 - 32):
        w = randn(n, k, dtype=BF16, scale=0.05)
        got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(w.to(DEV)), None, None, F32, packed_shape=(n, k))
        close(got, ref_gemm(x, w), atol=3e-5 * math.sqrt(k), rtol=1e-5, what=f"wide n={n}")
    for inner in (edge * 16, edge * 16 - 16):
        w = randn(2 * inner, k, dtype=BF16, scale=0.05)
        gu = x.double() @ w.double().T
        g, u = gu[:, :inner], gu[:, inner:]
        got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(w.to(DEV), True), None, None, F32, gated=True,
                            packed_shape=(2 * inner, k))
        close(got, g / (1.0 + torch.exp(-g)) * u, atol=1e-4 * math.sqrt(k), rtol=1e-4, what=f"wide gated {inner}")


@pytest.mark.parametrize("t", [1, 8, 16, 17, 40, 64, 65, 130, 300])
@pytest.mark.parametrize("n, k", [(100, 96), (224, 200), (3584, 512), (264, 2368), (72, 18944 // 8)])
@pytest.mark.parametrize("packed", [False, True])
def test_gemm_bf16_partial_slices_add_up(t, n, k, packed):
    """The product in K slices (packed weights: the stream kernel up to 64 rows, the tiled kernel
    beyond; row-major weights: the kernel whose waves split K): the slices add up to x w^T, and
    the consumers that add them give the fused results."""
    from sonicboom_amd import ops
    x, w = randn(t, k, dtype=BF16), randn(n, k, dtype=BF16, scale=0.05)
    wd = w.to(DEV)
    partial = ops.gemm_bf16_partial(x.to(DEV), ops.pack_weight(wd) if packed else wd,
                                    packed_shape=(n, k) if packed else None)
    if t > 64 and (not packed or partial is None):
        assert partial is None          # no cut that pays: the caller takes the whole product
        return
    assert partial is not None and partial.shape[1:] == (t, n) and 1 <= partial.shape[0] <= 8
    assert t <= 64 or partial.shape[0] > 1
    close(partial.double().sum(0), ref_gemm(x, w), atol=3e-5 * math.sqrt(k), rtol=1e-5, what="sum of the slices")
    if n % 4 == 0:
        resid, bias = randn(t, n), randn(n, scale=0.1)
        rd = resid.to(DEV)
        ops.reduce_resid_norm(partial, bias.to(DEV), rd, None, 1e-6, None)
        close(rd, ref_gemm(x, w, bias, resid), atol=3e-5 * math.sqrt(k), rtol=1e-5, what="slices + bias + residual")


def test_gemm_bf16_partial_in_big_tiles():
    """Two thousand rows against a narrow matrix with a long inner size: 56 tiles of 256 x 256 with
    K cut in four fill the GPU where 224 tiles of 128 x 128 would multiply whole.  The slices add
    up to the product (sampled rows against float64, all of it against the whole product), and
    the pass that adds them gives product + bias + residual and the norm of that."""
    from sonicboom_amd import ops
    t, n, k = 2048, 1792, 18944
    x, w = randn(t, k, dtype=BF16), randn(n, k, dtype=BF16, scale=0.02)
    xd, wp = x.to(DEV), ops.pack_weight(w.to(DEV))
    partial = ops.gemm_bf16_partial(xd, wp, packed_shape=(n, k))
    assert partial is not None and tuple(partial.shape) == (4, t, n)
    total = partial.double().sum(0)
    rows = [0, 1, 255, 256, 1000, 2047]
    close(total[rows], ref_gemm(x[rows], w), atol=3e-5 * math.sqrt(k), rtol=1e-5, what="sampled rows")
    whole = ops.gemm_bf16(xd, wp, None, None, F32, packed_shape=(n, k))
    close(total, whole.double().cpu(), atol=3e-5 * math.sqrt(k), rtol=1e-5, what="against the whole product")
    resid, bias, nw = randn(t, n), randn(n, scale=0.1), 1.0 + randn(n, scale=0.1)
    rd = resid.to(DEV)
    normed = ops.reduce_resid_norm(partial, bias.to(DEV), rd, nw.to(DEV), 1e-5, F32)
    want = whole.double().cpu() + bias.double() + resid.double()
    close(rd, want, atol=3e-5 * math.sqrt(k), rtol=1e-5, what="slices + bias + residual")
    want_n = want / torch.sqrt((want * want).mean(-1, keepdim=True) + 1e-5) * nw.double()
    close(normed, want_n, atol=1e-4, rtol=1e-4, what="and the norm")
    # a short inner size: the pass over four slices would cost more than the cut saves
    assert ops.gemm_bf16_partial(xd[:, :1024].contiguous(), ops.pack_weight(w[:, :1024].contiguous().to(DEV)),
                                 packed_shape=(n, 1024)) is None


@pytest.mark.parametrize("which, waves, slices", [("stream", 4, 1), ("stream", 5, 3), ("stream", 7, 8), ("stream", 8, 5),
                                                  ("tiled", 0, 0), ("skinny", 0, 0)])
@pytest.mark.parametrize("t", [3, 16, 33, 64])
@pytest.mark.parametrize("n, k", [(100, 96), (1000, 520), (264, 2368), (72, 4744)])
def test_gemm_bf16_partial_every_kernel(which, waves, slices, t, n, k):
    """Each kernel that can cut K, at forced cuts: slices that end inside a staged chunk of 256 k
    and inside a k-step, more slices asked for than K has chunks, columns that end inside a
    tile."""
    from sonicboom_amd import ops
    x, w = randn(t, k, dtype=BF16), randn(n, k, dtype=BF16, scale=0.05)
    with ops.gemm_few_rows_kernel(which, waves, slices):
        partial = ops.gemm_bf16_partial(x.to(DEV), ops.pack_weight(w.to(DEV)), packed_shape=(n, k))
    assert partial is not None and partial.shape[1:] == (t, n) and 1 <= partial.shape[0] <= 8
    if which == "stream" and slices:
        assert partial.shape[0] <= slices
    close(partial.double().sum(0), ref_gemm(x, w), atol=3e-5 * math.sqrt(k), rtol=1e-5, what=f"{which}: sum of the slices")


def test_gemm_bf16_refuses_what_it_cannot_take():
    from sonicboom_amd import ops
    x, w = randn(4, 100, dtype=BF16).to(DEV), randn(8, 100, dtype=BF16).to(DEV)
    assert ops.gemm_bf16(x, w, None, None, F32) is None          # inner size not a multiple of 8
    want = ref_gemm(x.cpu(), w.cpu())
    close(ops.gemm_plain(x, w, None, None, F32), want, atol=1e-3, rtol=1e-5)


@pytest.mark.parametrize("dtype", [F32, BF16])
def test_silu_mul_add_cast(dtype):
    from sonicboom_amd import ops
    gu = randn(9, 2 * 77, scale=3.0)
    gu[0, 0], gu[0, 1], gu[0, 2] = 0.0, 1.0, -100.0
    want = plain.silu(gu[:, :77].numpy()) * gu[:, 77:].numpy()
    got = ops.silu_mul(gu.to(DEV), dtype)
    close(got, want, atol=1e-6 if dtype == F32 else 2e-2, rtol=1e-6 if dtype == F32 else 8e-3)
    # silu(0) = 0, silu(1) = 0.7310586 (/root/reference/tests/core/test_nn.cpp:52-66)
    one = ops.silu_mul(torch.tensor([[0.0, 1.0, 1.0, 1.0]], device=DEV), F32).cpu()
    assert one[0, 0] == 0.0 and abs(one[0, 1].item() - 0.7310586) < 1e-6
    resid = randn(5, 33)
    y = randn(5, 33, dtype=dtype, seed=3)
    r = resid.to(DEV)
    ops.add_into(r, y.to(DEV))
    assert torch.equal(r.cpu(), resid + y.float())
    c = ops.cast(resid.to(DEV), BF16)
    assert torch.equal(c.cpu(), resid.to(BF16))


def make_cache(n_pages, heads_kv, head_dim, dtype, fill=float("nan")):
    """Keys [pages, heads, 64, d] and values [pages, heads, d, 64], filled with NaN: whatever a
    kernel reads beyond what was stored shows in its result.  Within a row the cache keeps its own
    order of elements; the tests read and write through sonicboom_amd.cache.layout."""
    k = torch.full((n_pages, heads_kv, 64, head_dim), fill, dtype=dtype, device=DEV)
    v = torch.full((n_pages, heads_kv, head_dim, 64), fill, dtype=dtype, device=DEV)
    return k, v


@pytest.mark.parametrize("hq, hkv, hd, rot", [(4, 2, 16, 0), (3, 1, 32, 0), (5, 5, 48, 0), (2, 1, 64, 32), (8, 2, 128, 0)])
@pytest.mark.parametrize("dtype", [F32, BF16])
def test_rope_kv_store(hq, hkv, hd, rot, dtype):
    """Rotation against the plain rope; keys and values land where the page table says."""
    from sonicboom_amd import ops
    base = 10000.0
    n = 11
    qkv = randn(n, (hq + 2 * hkv) * hd)
    pos = torch.tensor([0, 1, 2, 63, 64, 65, 130, 7, 200, 1000, 5], dtype=torch.int32)
    seq = torch.tensor([0, 0, 0, 0, 0, 0, 0, 1, 1, 1, 1], dtype=torch.int32)   # row -> sequence
    pos[7:] = torch.tensor([3, 64, 127, 128])
    # scattered physical pages, different per sequence
    table = torch.tensor([[5, 2, 7], [1, 6, 3]], dtype=torch.int32)
    kc, vc = make_cache(8, hkv, hd, dtype)
    dims = rot or hd
    ff = (1.0 + torch.arange(dims // 2, dtype=F32) / 7.0) if rot else None
    log_base = np.log(np.float32(base)).astype(np.float32)
    inv = np.exp((np.float32(-2.0) * np.arange(dims // 2, dtype=np.float32) / np.float32(dims)).astype(np.float32)
                 * log_base).astype(np.float32)
    q = ops.rope_kv_store(qkv.to(DEV), dtype, torch.from_numpy(inv).to(DEV), None if ff is None else ff.to(DEV),
                          dims, pos.to(DEV), seq.to(DEV), kc, vc, table.to(DEV), hq, hkv, hd)
    qw, kvw = hq * hd, hkv * hd
    ffn = None if ff is None else ff.numpy()
    want_q = plain.rope_neox(qkv[:, :qw].numpy(), pos.numpy(), hd, base, rot, ffn)
    want_k = plain.rope_neox(qkv[:, qw:qw + kvw].numpy(), pos.numpy(), hd, base, rot, ffn)
    tol = dict(atol=2e-6, rtol=1e-5) if dtype == F32 else dict(atol=2e-2, rtol=8e-3)
    close(q, want_q, what="q", **tol)
    for r in range(n):
        page = table[seq[r], pos[r] // 64]
        got_k = layout.get_key(kc, int(page), int(pos[r]) % 64).reshape(-1)
        got_v = layout.get_value(vc, int(page), int(pos[r]) % 64).reshape(-1)
        close(got_k, want_k[r], what=f"k row {r}", **tol)
        close(got_v, qkv[r, qw + kvw:].to(dtype).float(), atol=0, rtol=0, what=f"v row {r}")
    # nothing else was written
    assert torch.isnan(kc.float()).sum().item() == kc.numel() - n * kvw


@pytest.mark.parametrize("hq, hkv, hd, rot", [(7, 1, 48, 0), (28, 4, 128, 0), (3, 3, 64, 32)])
def test_rope_kv_store_many_rows_equals_few_rows(hq, hkv, hd, rot):
    """A prompt of 700 rows in one call (all heads of a row in one block) gives bitwise what the
    same rows give in calls of 100 (groups of four heads)."""
    from sonicboom_amd import ops
    n = 700
    qkv = randn(n, (hq + 2 * hkv) * hd).to(DEV)
    bias = randn((hq + 2 * hkv) * hd, scale=0.1, seed=3).to(DEV)
    pos = torch.arange(n, dtype=torch.int32, device=DEV)
    seq = torch.zeros(n, dtype=torch.int32, device=DEV)
    table = torch.tensor([[4, 9, 1, 7, 3, 10, 0, 6, 2, 8, 5]], dtype=torch.int32, device=DEV)
    dims = rot or hd
    inv = torch.exp(-2.0 * torch.arange(dims // 2, dtype=F32) / dims * math.log(1e6)).to(DEV)
    results = []
    for step in (n, 100):
        kc, vc = make_cache(11, hkv, hd, BF16, fill=0.0)
        qs = [ops.rope_kv_store(qkv[r0:r0 + step], BF16, inv, None, dims, pos[r0:r0 + step], seq[r0:r0 + step], kc, vc,
                                table, hq, hkv, hd, bias=bias) for r0 in range(0, n, step)]
        results.append((torch.cat(qs), kc, vc))
    for a, b in zip(*results):
        assert torch.equal(a, b)
    want_q = plain.rope_neox((qkv.cpu() + bias.cpu())[:, :hq * hd].numpy(), pos.cpu().numpy(), hd, 1e6, rot, None)
    close(results[0][0], want_q, atol=2e-2, rtol=8e-3, what="q of the long prompt")


@pytest.mark.parametrize("hq, hkv, hd, rot", [(7, 1, 48, 0), (28, 4, 128, 0), (3, 3, 64, 32), (5, 2, 80, 0), (2, 0, 32, 0)])
@pytest.mark.parametrize("rotate", [True, False])
@pytest.mark.parametrize("in_dtype", [F32, BF16])
def test_rope_kv_store_rows_eight_pairs_at_a_time(hq, hkv, hd, rot, rotate, in_dtype):
    """A prompt step's qkv rows (float32 as the engine has them, or bfloat16; no slices, no bias)
    go through the kernel that moves eight pairs per load and store: bitwise what the same rows
    give in calls of 100, which take the element-wise kernel; with a partial rotary width,
    without rotation, and for a layer that stores no keys."""
    from sonicboom_amd import ops
    n = 700
    qkv = randn(n, (hq + 2 * hkv) * hd, dtype=in_dtype).to(DEV)
    pos = (torch.arange(n, dtype=torch.int32) * 3 % 701).to(DEV)
    seq = torch.zeros(n, dtype=torch.int32, device=DEV)
    table = torch.tensor([[4, 9, 1, 7, 3, 10, 0, 6, 2, 8, 5]], dtype=torch.int32, device=DEV)
    dims = rot or hd
    inv = torch.exp(-2.0 * torch.arange(dims // 2, dtype=F32) / dims * math.log(1e6)).to(DEV) if rotate else None
    results = []
    for step in (n, 100):
        kc, vc = make_cache(11, max(hkv, 1), hd, BF16, fill=0.0)
        qs = [ops.rope_kv_store(qkv[r0:r0 + step], BF16, inv, None, dims, pos[r0:r0 + step], seq[r0:r0 + step], kc, vc,
                                table, hq, hkv, hd) for r0 in range(0, n, step)]
        results.append((torch.cat(qs), kc, vc))
    for a, b in zip(*results):
        assert torch.equal(a, b)
    if rotate:
        want_q = plain.rope_neox(qkv.float().cpu()[:, :hq * hd].numpy(), pos.cpu().numpy(), hd, 1e6, rot, None)
        close(results[0][0], want_q, atol=2e-2, rtol=8e-3, what="q of the long prompt")
    else:
        assert torch.equal(results[0][0], qkv[:, :hq * hd].to(BF16))


@pytest.mark.parametrize("hq, hkv, hd, rot", [(28, 4, 128, 0), (3, 3, 64, 32), (5, 2, 80, 0)])
@pytest.mark.parametrize("slices", [2, 3, 5])
@pytest.mark.parametrize("in_dtype", [F32, BF16])
def test_rope_kv_store_rows_in_slices_with_a_bias(hq, hkv, hd, rot, slices, in_dtype):
    """The same kernel takes a prompt's qkv rows as K slices of the product with the bias still to
    add (what the sliced product of a few hundred rows leaves): slices added in ascending order,
    then the bias, bitwise as the element-wise kernel does it in calls of 100 rows, and the sum is
    the plain rotation of the summed rows."""
    from sonicboom_amd import ops
    n, w = 700, (hq + 2 * hkv) * hd
    parts = randn(slices, n, w, dtype=in_dtype).to(DEV)
    bias = randn(w, scale=0.1, seed=3).to(DEV)
    pos = (torch.arange(n, dtype=torch.int32) * 3 % 701).to(DEV)
    seq = torch.zeros(n, dtype=torch.int32, device=DEV)
    table = torch.tensor([[4, 9, 1, 7, 3, 10, 0, 6, 2, 8, 5]], dtype=torch.int32, device=DEV)
    dims = rot or hd
    inv = torch.exp(-2.0 * torch.arange(dims // 2, dtype=F32) / dims * math.log(1e6)).to(DEV)
    results = []
    for step in (n, 100):
        kc, vc = make_cache(11, hkv, hd, BF16, fill=0.0)
        qs = [ops.rope_kv_store(parts[:, r0:r0 + step].contiguous(), BF16, inv, None, dims, pos[r0:r0 + step],
                                seq[r0:r0 + step], kc, vc, table, hq, hkv, hd, bias=bias) for r0 in range(0, n, step)]
        results.append((torch.cat(qs), kc, vc))
    for a, b in zip(*results):
        assert torch.equal(a, b)
    rows = parts.float().sum(dim=0).cpu() + bias.cpu()
    want_q = plain.rope_neox(rows[:, :hq * hd].numpy(), pos.cpu().numpy(), hd, 1e6, rot, None)
    close(results[0][0], want_q, atol=3e-2, rtol=8e-3, what="q of the long prompt")
    page, slot = int(table[0, int(pos[650]) // 64]), int(pos[650]) % 64
    close(layout.get_value(results[0][2], page, slot).reshape(-1), rows[650, (hq + hkv) * hd:].to(BF16).float(),
          atol=2e-2, rtol=8e-3, what="a value row")


def test_rope_reference_vectors():
    """/root/reference/tests/core/test_nn.cpp:221-290: position 0 is the identity; with
    head size 2 and an angle of pi/2, [1,0] turns into [0,1]; pairs are (i, i+half)."""
    from sonicboom_amd import ops
    kc, vc = make_cache(1, 1, 4, F32)
    table = torch.zeros((1, 1), dtype=torch.int32, device=DEV)
    z = torch.zeros(1, dtype=torch.int32, device=DEV)
    x = torch.tensor([[0.5, -1.25, 2.0, 3.5] * 3], device=DEV)
    inv = torch.tensor([1.0, 0.01], device=DEV)
    q = ops.rope_kv_store(x, F32, inv, None, 4, z, z, kc, vc, table, 1, 1, 4)
    assert torch.equal(q.cpu(), x[:, :4].cpu())
    # angle pi/2 for both pairs at position 1: (x0, x2) -> (-x2, x0), (x1, x3) -> (-x3, x1)
    inv = torch.full((2,), math.pi / 2, device=DEV)
    one = torch.ones(1, dtype=torch.int32, device=DEV)
    x = torch.tensor([[1.0, 0.0, 2.0, 3.0] * 3], device=DEV)
    q = ops.rope_kv_store(x, F32, inv, None, 4, one, z, kc, vc, table, 1, 1, 4).cpu()
    assert torch.allclose(q, torch.tensor([[-2.0, -3.0, 1.0, 0.0]]), atol=1e-6)
    # freq_factors: a huge divisor freezes its pair (test_nn.cpp:272-289)
    ff = torch.tensor([1.0, 1e30], device=DEV)
    q = ops.rope_kv_store(x, F32, inv, ff, 4, one, z, kc, vc, table, 1, 1, 4).cpu()
    assert torch.allclose(q, torch.tensor([[-2.0, 0.0, 1.0, 3.0]]), atol=1e-5)


def fill_cache_from(keys, values, table, dtype):
    """keys/values: list per sequence of [len, hkv, hd] float tensors -> paged caches."""
    hkv, hd = keys[0].shape[1:]
    n_pages = int(table.max()) + 1
    kc, vc = make_cache(n_pages, hkv, hd, dtype)
    for s, (k, v) in enumerate(zip(keys, values)):
        for p in range(k.shape[0]):
            page = table[s, p // 64]
            layout.put_key(kc, int(page), p % 64, k[p])
            layout.put_value(vc, int(page), p % 64, v[p])
    return kc, vc


ATTN_SHAPES = [(4, 2, 16), (3, 1, 32), (5, 5, 48), (6, 2, 80), (8, 2, 128), (2, 1, 256)]


@pytest.mark.parametrize("hq, hkv, hd", ATTN_SHAPES)
@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("window", [0, 70])
def test_attention_plain_kernel(hq, hkv, hd, dtype, window):
    from sonicboom_amd import ops
    lens = [150, 3]
    table = torch.tensor([[4, 0, 2], [1, 3, 5]], dtype=torch.int32)
    keys = [randn(n, hkv, hd, seed=s).to(dtype).float() for s, n in enumerate(lens)]
    vals = [randn(n, hkv, hd, seed=9 + s).to(dtype).float() for s, n in enumerate(lens)]
    kc, vc = fill_cache_from(keys, vals, table, dtype)
    # rows: a few positions of sequence 0 (first, page edges, last), all of sequence 1
    rows = [(0, 0), (0, 63), (0, 64), (0, 100), (0, 149), (1, 0), (1, 1), (1, 2)]
    q = randn(len(rows), hq * hd, seed=5).to(dtype)
    scale = 1.0 / math.sqrt(hd)
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32)
    seq = torch.tensor([s for s, _ in rows], dtype=torch.int32)
    got = ops.attention_plain(q.to(DEV), kc, vc, table.to(DEV), pos.to(DEV), seq.to(DEV), hq, hkv, hd, scale, window)
    for r, (s, p) in enumerate(rows):
        n = lens[s]
        want = plain.attention(q[r:r + 1].float().numpy(), keys[s].reshape(n, -1).numpy(),
                               vals[s].reshape(n, -1).numpy(), [p], np.arange(n), hq, hkv, hd, scale,
                               causal=True, window=window)
        tol = dict(atol=3e-6, rtol=2e-5) if dtype == F32 else dict(atol=2e-2, rtol=1e-2)
        close(got[r:r + 1], want, what=f"row {r} (seq {s}, pos {p})", **tol)


@pytest.mark.parametrize("hq, hkv, hd", [(4, 2, 16), (3, 1, 20), (2, 1, 256)])
@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("window", [0, 1, 64, 65, 130])
@pytest.mark.parametrize("keys", [50, 64, 100, 240, 600])
def test_attention_plain_waves_of_a_block(hq, hkv, hd, dtype, window, keys):
    """However many of a block's waves share a row's keys (the table's width and the window say how many there may be,
    the count of rows how many the launcher likes), the bits are the same."""
    from sonicboom_amd import ops
    pages = (keys + 63) // 64
    table = torch.randperm(pages, generator=torch.Generator().manual_seed(1)).int()[None]
    kc, vc = (randn(pages, hkv, 64, hd, seed=2).to(dtype).to(DEV), randn(pages, hkv, hd, 64, seed=3).to(dtype).to(DEV))
    rows = [0, 1, min(63, keys - 1), min(64, keys - 1), keys // 2, keys - 1]
    outs = []
    for extra, times in ((0, 1), (3, 1), (9, 1), (0, 200)):
        t = torch.cat([table, torch.full((1, extra), -1, dtype=torch.int32)], 1).to(DEV)
        q = randn(len(rows), hq * hd, seed=4).to(dtype).repeat(times, 1).to(DEV)
        pos = torch.tensor(rows * times, dtype=torch.int32, device=DEV)
        outs.append(ops.attention_plain(q, kc, vc, t, pos, torch.zeros_like(pos), hq, hkv, hd, hd ** -0.5, window))
    assert all(torch.equal(outs[0], o[:len(rows)]) and torch.equal(o[-len(rows):], outs[0]) for o in outs)


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("hd", [20, 64])
@pytest.mark.parametrize("gone", [[64], [70], [64, 130], list(range(64, 128)), list(range(128, 140))])
def test_attention_plain_scores_out_of_range(hd, dtype, gone):
    """Keys whose score is minus infinity weigh nothing, alone in a chunk of keys or all of it, in the last chunk or before."""
    from sonicboom_amd import ops
    hq, hkv, n = 4, 2, 140
    rows = [64, 70, 127, 128, 139]
    q, k, v = randn(len(rows), hq, hd), randn(n, hkv, hd, seed=1), randn(n, hkv, hd, seed=2)
    q[..., 3], k[..., 3] = 1e25, 0.0
    k[gone, :, 3] = -1e25                      # the product of the two lies below the float32 range
    q, k, v = q.to(dtype), k.to(dtype), v.to(dtype)
    table = torch.tensor([[2, 0, 1]], dtype=torch.int32)
    kc, vc = fill_cache_from([k], [v], table, dtype)
    got = ops.attention_plain(q.reshape(len(rows), hq * hd).to(DEV), kc, vc, table.to(DEV), torch.tensor(rows, dtype=torch.int32).to(DEV),
                              torch.zeros(len(rows), dtype=torch.int32).to(DEV), hq, hkv, hd, hd ** -0.5, 0)
    kept = [j for j in range(n) if j not in gone]
    want = torch.zeros(len(rows), hq, hd, dtype=torch.float64)
    for i, pos in enumerate(rows):
        js = [j for j in kept if j <= pos]
        for h in range(hq):
            p = torch.softmax(k[js, h // 2].double() @ q[i, h].double() * hd ** -0.5, 0)
            want[i, h] = p @ v[js, h // 2].double()
    close(got, want.reshape(len(rows), hq * hd), atol=2e-5 if dtype == F32 else 2e-2, rtol=1e-5 if dtype == F32 else 1e-2)


def attention_case(hq, hkv, hd, lens, rows_per_seq, window, seed=0):
    """Random bf16 keys, values and queries for sequences of ``lens`` tokens on scattered pages;
    ``rows_per_seq[s]`` lists the positions of sequence s that ask.  Returns device operands and the
    plain result per row."""
    n_seq = len(lens)
    width = max((n + 63) // 64 for n in lens)
    perm = torch.randperm(n_seq * width + 3, generator=torch.Generator().manual_seed(seed))
    table = torch.full((n_seq, width), -1, dtype=torch.int32)
    it = iter(perm.tolist())
    for s_, n in enumerate(lens):
        for pg in range((n + 63) // 64):
            table[s_, pg] = next(it)
    keys = [randn(n, hkv, hd, seed=seed + s_).to(BF16).float() for s_, n in enumerate(lens)]
    vals = [randn(n, hkv, hd, seed=seed + 50 + s_).to(BF16).float() for s_, n in enumerate(lens)]
    hkv_, hd_ = keys[0].shape[1:]
    kc, vc = make_cache(n_seq * width + 3, hkv_, hd_, BF16)
    for s_, (k, v) in enumerate(zip(keys, vals)):
        for p in range(k.shape[0]):
            page = table[s_, p // 64]
            layout.put_key(kc, int(page), p % 64, k[p])
            layout.put_value(vc, int(page), p % 64, v[p])
    rows = [(s_, p) for s_, ps in enumerate(rows_per_seq) for p in ps]
    q = randn(len(rows), hq * hd, seed=seed + 7).to(BF16)
    scale = 1.0 / math.sqrt(hd)
    want = []
    for r, (s_, p) in enumerate(rows):
        n = lens[s_]
        want.append(plain.attention(q[r:r + 1].float().numpy(), keys[s_].reshape(n, -1).numpy(),
                                    vals[s_].reshape(n, -1).numpy(), [p], np.arange(n), hq, hkv, hd, scale,
                                    causal=True, window=window))
    return q, kc, vc, table, rows, scale, np.concatenate(want, axis=0)


# (groups of 7, 5 and 8 query heads per kv head run prefill with eight waves a block: one, three
# and no wave without a head; the last shape makes a second block of one head and three such waves)
# (from (8, 2, 128) on: every wave of a block of four has a head and all waves share the loads that
# bring a page in; heads of more than 128 in blocks of eight waves: sixteen heads in two blocks,
# five heads and three waves without one, eight heads; groups of one and two heads at usual head sizes)
MFMA_SHAPES = [(4, 2, 16), (3, 1, 32), (5, 5, 48), (6, 2, 80), (28, 4, 128), (2, 1, 256), (40, 2, 64), (10, 2, 128),
               (16, 2, 64), (8, 2, 128), (4, 1, 256), (16, 1, 192), (10, 2, 160), (8, 1, 144), (3, 3, 128), (4, 2, 64),
               (12, 1, 96)]


@pytest.mark.parametrize("hq, hkv, hd", MFMA_SHAPES)
@pytest.mark.parametrize("window", [0, 70])
def test_attention_decode_matrix_cores(hq, hkv, hd, window):
    """One row per sequence, lengths on both sides of page and chunk (4 pages) edges."""
    from sonicboom_amd import ops
    lens = [1, 2, 64, 65, 255, 256, 257, 700]
    q, kc, vc, table, rows, scale, want = attention_case(hq, hkv, hd, lens, [[n - 1] for n in lens], window)
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32)
    got = ops.attention_decode_mfma(q.to(DEV), kc, vc, table.to(DEV), pos.to(DEV), hq, hkv, hd, scale, window)
    close(got, want, atol=1.5e-2, rtol=1e-2, what="decode")
    for _ in range(3):                       # launch after launch, the same bits
        again = ops.attention_decode_mfma(q.to(DEV), kc, vc, table.to(DEV), pos.to(DEV), hq, hkv, hd, scale, window)
        assert torch.equal(got, again)


@pytest.mark.parametrize("window", [0, 100])
@pytest.mark.parametrize("longest", [300, 900])
def test_attention_decode_matrix_cores_many_sequences(window, longest):
    """Two hundred sequences: a block for every CU without cutting the rows, so each block takes
    its row whole (one chunk, a quarter of the table's width per wave, no merge kernel); lengths
    from one key to many pages, with and without a window."""
    from sonicboom_amd import ops
    hq, hkv, hd = 8, 4, 32
    rng = np.random.default_rng(5)
    lens = [int(n) for n in rng.integers(1, longest, size=200)]
    lens[:4] = [1, 64, 65, longest]
    q, kc, vc, table, rows, scale, want = attention_case(hq, hkv, hd, lens, [[n - 1] for n in lens], window, seed=9)
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32)
    got = ops.attention_decode_mfma(q.to(DEV), kc, vc, table.to(DEV), pos.to(DEV), hq, hkv, hd, scale, window)
    close(got, want, atol=1.5e-2, rtol=1e-2, what="decode, 200 sequences")


@pytest.mark.parametrize("window", [0, 300])
@pytest.mark.parametrize("n_seqs, longest", [(30, 2000), (12, 5000), (3, 9000), (70, 1500)])
def test_attention_decode_matrix_cores_long_rows_of_unequal_length(window, n_seqs, longest):
    """Rows long enough for the launcher to deal several pages to a wave and cut the rows into
    chunks of its own choosing; lengths from one key to thousands in one batch, so that chunks
    are full, partly filled and empty side by side.  (70 sequences on 4 kv heads: a few blocks
    more than the GPU has CUs, for which the launcher takes smaller chunks.)"""
    from sonicboom_amd import ops
    hq, hkv, hd = 8, 4, 64
    rng = np.random.default_rng(n_seqs)
    lens = [int(n) for n in rng.integers(1, longest, size=n_seqs)]
    lens[0], lens[-1] = longest, 1
    q, kc, vc, table, rows, scale, want = attention_case(hq, hkv, hd, lens, [[n - 1] for n in lens], window, seed=21)
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32)
    got = ops.attention_decode_mfma(q.to(DEV), kc, vc, table.to(DEV), pos.to(DEV), hq, hkv, hd, scale, window)
    close(got, want, atol=1.5e-2, rtol=1e-2, what=f"decode, {n_seqs} rows up to {longest} keys")


@pytest.mark.parametrize("hq, hkv, hd", [(4, 2, 16), (5, 5, 48), (14, 2, 64), (40, 2, 64), (6, 2, 80), (28, 4, 128)])
@pytest.mark.parametrize("window", [0, 70])
@pytest.mark.parametrize("longest", [257, 320, 448, 449, 512, 513])
def test_attention_decode_of_rows_that_one_block_takes_whole(hq, hkv, hd, window, longest):
    """Heads of up to 128 numbers, tables of five to eight pages (and of nine: chunks again): lengths around the edges of
    pages and of the eight waves, page numbers outside the cache behind the window."""
    from sonicboom_amd import ops
    lens = [1, 64, 65, 256, 257, longest]
    q, kc, vc, table, rows, scale, want = attention_case(hq, hkv, hd, lens, [[n - 1] for n in lens], window, seed=4)
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32)
    if window:
        table[-1, 0] = -1
        table[-1, 1] = kc.shape[0] + 5
    got = ops.attention_decode_mfma(q.to(DEV), kc, vc, table.to(DEV), pos.to(DEV), hq, hkv, hd, scale, window)
    close(got, want, atol=1.5e-2, rtol=1e-2, what="decode, whole rows")
    with ops.attention_decode_pages_per_wave(hd, 1):
        chunks = ops.attention_decode_mfma(q.to(DEV), kc, vc, table.to(DEV), pos.to(DEV), hq, hkv, hd, scale, window)
    # the same sums of float32 numbers in another order, then one rounding to bfloat16
    close(got, chunks.float().cpu(), atol=2.0 ** -7, rtol=2.0 ** -7, what="against chunks of four pages")


@pytest.mark.parametrize("hq, hkv, hd", [(4, 2, 16), (5, 5, 48), (6, 2, 80), (28, 4, 128), (40, 2, 64)])
@pytest.mark.parametrize("window", [0, 70, 1000])
@pytest.mark.parametrize("pages", [1, 2, 4, 8])
def test_attention_decode_pages_per_wave(hq, hkv, hd, window, pages):
    """Every way of dealing pages to waves (one page each, or 2, 4, 8 in a row with the next half
    page in flight), on lengths around page, wave and chunk edges, a long row, a window that
    starts inside a later chunk, and a table with a hole: a page number outside the cache in a
    page that the window has left behind."""
    from sonicboom_amd import ops
    lens = [1, 64, 65, 129, 256, 257, 513, 700, 2100]
    q, kc, vc, table, rows, scale, want = attention_case(hq, hkv, hd, lens, [[n - 1] for n in lens], window, seed=4)
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32)
    if window:
        table[-1, 0] = -1                     # the cache gives such pages back
        table[-1, 1] = kc.shape[0] + 5
    with ops.attention_decode_pages_per_wave(hd, pages):
        got = ops.attention_decode_mfma(q.to(DEV), kc, vc, table.to(DEV), pos.to(DEV), hq, hkv, hd, scale, window)
        close(got, want, atol=1.5e-2, rtol=1e-2, what=f"decode, {pages} pages per wave")
        again = ops.attention_decode_mfma(q.to(DEV), kc, vc, table.to(DEV), pos.to(DEV), hq, hkv, hd, scale, window)
        assert torch.equal(got, again)


@pytest.mark.parametrize("hq, hkv, hd", MFMA_SHAPES)
@pytest.mark.parametrize("window", [0, 70])
def test_attention_prefill_matrix_cores(hq, hkv, hd, window):
    """Whole prompts of unequal lengths, and a continuation on top of cached keys."""
    from sonicboom_amd import ops
    lens = [1, 17, 64, 150, 200]
    starts = [0, 0, 0, 0, 120]           # the last sequence has 120 keys cached and brings 80 rows
    rows_per_seq = [list(range(s0, n)) for s0, n in zip(starts, lens)]
    q, kc, vc, table, rows, scale, want = attention_case(hq, hkv, hd, lens, rows_per_seq, window, seed=3)
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32)
    # tiles of 16 rows, of the height that suits the group (64 and 32 rows for groups of one and two
    # heads), and of 32 rows where the kernel has its form for long prompts
    for height in sorted({16, ops.attention_row_tile(hq, hkv, hd)} | ({32} if ops.attention_tall_ok(hq, hkv, hd) else set())):
        tiles, row0 = [], 0
        for s_, ps in enumerate(rows_per_seq):
            for r0 in range(0, len(ps), height):
                tiles.append((row0 + r0, min(height, len(ps) - r0), s_, 0))
            row0 += len(ps)
        tiles = torch.tensor(tiles, dtype=torch.int32)
        got = ops.attention_prefill_mfma(q.to(DEV), kc, vc, table.to(DEV), pos.to(DEV), tiles.to(DEV), hq, hkv, hd,
                                         scale, window, tile_rows=height)
        close(got, want, atol=1.5e-2, rtol=1e-2, what=f"prefill, tiles of {height} rows")
    assert ops.attention_row_tile(hq, hkv, hd) == (64 if hq == hkv else 32 if hq == 2 * hkv else 16)
    assert ops.attention_tall_ok(hq, hkv, hd) == (hq >= 3 * hkv and hd % 32 == 0 and hd <= 128)
    assert ops.attention_row_tiles(hq, hkv, hd) == ((16, 32) if ops.attention_tall_ok(hq, hkv, hd)
                                                    else (ops.attention_row_tile(hq, hkv, hd),))
    if hq > 2 * hkv:
        with pytest.raises(ops.KernelLibraryError, match="do not suit"):
            ops.attention_prefill_mfma(q.to(DEV), kc, vc, table.to(DEV), pos.to(DEV), tiles.to(DEV), hq, hkv, hd,
                                       scale, window, tile_rows=64)


def test_attention_reference_vectors():
    """/root/reference/tests/core/test_nn.cpp:402-495: one key copies its value; causal
    2x2 gives [2, 3]; GQA maps 4 query heads onto 2 kv heads; window 2 drops key 0;
    scale 1 and 0.5 give 1.0360 and 1.2384."""
    from sonicboom_amd import ops

    def run(q, k, v, hq, hkv, hd, scale, window=0):
        n = len(k)
        keys = [torch.tensor(k, dtype=F32).reshape(n, hkv, hd)]
        vals = [torch.tensor(v, dtype=F32).reshape(n, hkv, hd)]
        table = torch.zeros((1, 1), dtype=torch.int32)
        # pad the head to the kernels' smallest size by zero columns: scores are unchanged
        kc, vc = fill_cache_from(keys, vals, table, F32)
        qt = torch.tensor(q, dtype=F32).reshape(-1, hq * hd)
        pos = torch.arange(qt.shape[0], dtype=torch.int32)
        seq = torch.zeros(qt.shape[0], dtype=torch.int32)
        return ops.attention_plain(qt.to(DEV), kc, vc, table.to(DEV), pos.to(DEV), seq.to(DEV), hq, hkv, hd,
                                   scale, window).cpu()

    assert torch.allclose(run([[1.0, 0, 0, 0]], [[1.0, 0, 0, 0]], [[1.0, 2, 3, 4]], 1, 1, 4, 1.0),
                          torch.tensor([[1.0, 2, 3, 4]]), atol=1e-6)
    out = run([[1.0], [1.0]], [[1.0], [1.0]], [[2.0], [4.0]], 1, 1, 1, 1.0)
    assert torch.allclose(out.flatten(), torch.tensor([2.0, 3.0]), atol=1e-6)
    out = run([[1.0, 1, 1, 1]], [[1.0, 1.0]], [[1.0, 2.0]], 4, 2, 1, 1.0)
    assert torch.allclose(out.flatten(), torch.tensor([1.0, 1.0, 2.0, 2.0]), atol=1e-6)
    out = run([[1.0], [1.0], [1.0]], [[1.0], [1.0], [1.0]], [[1.0], [2.0], [4.0]], 1, 1, 1, 1.0, window=2)
    assert abs(out[2, 0].item() - 3.0) < 1e-6
    # q = 2 at the position of the second key; keys [2, 0], values [1, 3]
    for scale, want in ((1.0, 1.0360), (0.5, 1.2384)):
        out = run([[0.0], [2.0]], [[2.0], [0.0]], [[1.0], [3.0]], 1, 1, 1, scale)
        assert abs(out[1, 0].item() - want) < 1e-3


def test_a_far_key_among_hundreds_is_found():
    """One key far back is made to dominate: the output must be its value, whatever page it is on."""
    from sonicboom_amd import ops
    hq, hkv, hd, n = 4, 2, 32, 700
    keys = [randn(n, hkv, hd, scale=0.1)]
    vals = [randn(n, hkv, hd, seed=2)]
    q = randn(1, hq * hd, seed=4)
    table = torch.tensor([list(reversed(range(11)))], dtype=torch.int32)
    for far in (0, 63, 64, 389, 699):
        k = [keys[0].clone()]
        for h in range(hq):
            k[0][far, h // 2] = q[0, h * hd:(h + 1) * hd] * 40.0 if h % 2 == 0 else k[0][far, h // 2]
        kc, vc = fill_cache_from(k, vals, table, F32)
        out = ops.attention_plain(q.to(DEV), kc, vc, table.to(DEV), torch.tensor([n - 1], dtype=torch.int32, device=DEV),
                                  torch.zeros(1, dtype=torch.int32, device=DEV), hq, hkv, hd, 1.0, 0).cpu()
        for h in (0, 2):
            assert torch.allclose(out[0, h * hd:(h + 1) * hd], vals[0][far, h // 2], atol=1e-4), (far, h)


@pytest.mark.parametrize("hq, hkv, hd", [(14, 2, 128), (4, 2, 64), (3, 1, 32)])
@pytest.mark.parametrize("shape", ["climbing", "falling", "far key"])
def test_attention_matrix_cores_when_the_maximum_moves(hq, hkv, hd, shape):
    """Scores made to climb page after page (the running maximum has to follow, in steps), to
    fall from the first key on (it never moves again), or to peak at one key far back among
    hundreds of small ones: prefill rows and decode rows against the plain softmax."""
    from sonicboom_amd import ops
    n, group = 600, hq // hkv
    scale = 1.0 / math.sqrt(hd)
    keys = randn(n, hkv, hd, scale=0.05, seed=11)
    vals = randn(n, hkv, hd, seed=12)
    rows_pos = list(range(552, 600))                 # 552 keys cached, 48 rows asking
    q = randn(len(rows_pos), hq * hd, scale=0.05, seed=13)
    q.view(len(rows_pos), hq, hd)[:, :, 0] = 8.0      # every head looks along coordinate 0
    ramp = torch.arange(n, dtype=torch.float32) / n   # 0 .. 1 over the sequence
    rise = 56.0 / (8.0 * scale)                       # scores span about 56 (81 in log2 units)
    if shape == "climbing":
        keys[:, :, 0] = (ramp * rise)[:, None]
    elif shape == "falling":
        keys[:, :, 0] = ((1.0 - ramp) * rise)[:, None]
    else:
        keys[389, :, 0] = rise
    keys, vals, q = keys.to(BF16).float(), vals.to(BF16).float(), q.to(BF16)
    table = torch.tensor([[7, 2, 9, 4, 0, 5, 1, 8, 3, 6]], dtype=torch.int32)
    kc, vc = fill_cache_from([keys], [vals], table, BF16)
    want = plain.attention(q.float().numpy(), keys.reshape(n, -1).numpy(), vals.reshape(n, -1).numpy(), rows_pos,
                           np.arange(n), hq, hkv, hd, scale, causal=True, window=0)
    pos = torch.tensor(rows_pos, dtype=torch.int32)
    for height in (16, 32) if ops.attention_tall_ok(hq, hkv, hd) else (16,):
        tiles = torch.tensor([(r0, min(height, len(rows_pos) - r0), 0, 0) for r0 in range(0, len(rows_pos), height)],
                             dtype=torch.int32)
        got = ops.attention_prefill_mfma(q.to(DEV), kc, vc, table.to(DEV), pos.to(DEV), tiles.to(DEV), hq, hkv, hd,
                                         scale, 0, tile_rows=height)
        close(got, want, atol=1.5e-2, rtol=1e-2, what=f"prefill, {shape}, tiles of {height}")
    # the same rows as single decode rows of sequences that share the pages
    for r in (0, 17, 47):
        got1 = ops.attention_decode_mfma(q[r:r + 1].to(DEV), kc, vc, table.to(DEV), pos[r:r + 1].to(DEV), hq, hkv,
                                         hd, scale, 0)
        close(got1, want[r:r + 1], atol=1.5e-2, rtol=1e-2, what=f"decode row {r}, {shape}")
    if shape == "far key":
        # the far key takes all the weight: the output is its value
        v_far = vals[389].repeat_interleave(group, dim=0).reshape(1, -1)
        close(got[-1:], v_far.numpy(), atol=2e-2, rtol=1e-2, what="far key's value")


def _looking_along_zero(n, hq, hkv, hd, n_rows, seed):
    """Small random keys and queries whose coordinate 0 is large in the queries: a key whose
    coordinate 0 is raised takes all of a row's weight.  Returns keys, values, queries, the raise
    that puts one score 56 above the rest, and the scale."""
    scale = 1.0 / math.sqrt(hd)
    keys = randn(n, hkv, hd, scale=0.05, seed=seed)
    vals = randn(n, hkv, hd, seed=seed + 1)
    q = randn(n_rows, hq * hd, scale=0.05, seed=seed + 2)
    q.view(n_rows, hq, hd)[:, :, 0] = 8.0
    return keys.to(BF16).float(), vals.to(BF16).float(), q.to(BF16), 56.0 / (8.0 * scale), scale


@pytest.mark.parametrize("pages", [0, 1, 2, 4, 8])
def test_attention_decode_one_dominant_key_in_each_chunk(pages):
    """A row of 6,500 keys is cut into chunks of 4 x ``pages`` pages whose partial results a
    second kernel merges.  One key at a time is made to dominate: the first key of all, the first
    and last key of a wave's run of pages in a middle chunk, the first key of the second and of
    the last chunk, the row's own key and the one before it.  The output must be that key's
    value: a chunk or a wave's run that is dropped, merged twice or weighted wrongly shows at
    once, where random keys would move the output by less than the tolerance."""
    from sonicboom_amd import ops
    hq, hkv, hd, n = 8, 2, 64, 6500
    keys, vals, q, rise, scale = _looking_along_zero(n, hq, hkv, hd, 1, seed=31)
    width = (n + 63) // 64
    table = torch.randperm(width + 5, generator=torch.Generator().manual_seed(3))[:width].to(torch.int32)[None, :]
    kc, vc = fill_cache_from([keys], [vals], table, BF16)
    pos = torch.tensor([n - 1], dtype=torch.int32, device=DEV)
    run = max(pages, 1)                    # pages of a wave's run; a chunk is four runs
    last_chunk = ((n - 1) // 64 // (4 * run)) * 4 * run * 64
    spots = sorted({0, 4 * run * 64, (4 * run + 2 * run) * 64, (4 * run + 2 * run) * 64 - 1,
                    (4 * run + run) * 64 - 1, last_chunk, last_chunk - 1, n - 2, n - 1})
    group = hq // hkv
    with ops.attention_decode_pages_per_wave(hd, pages):
        for far in spots:
            page, slot = int(table[0, far // 64]), far % 64
            at = int(layout.key_positions(hd)[slot, 0])          # where element 0 of that key lies
            before = kc[page, :, slot, at].clone()
            kc[page, :, slot, at] = rise
            got = ops.attention_decode_mfma(q.to(DEV), kc, vc, table.to(DEV), pos, hq, hkv, hd, scale, 0)
            kc[page, :, slot, at] = before
            want = vals[far].repeat_interleave(group, dim=0).reshape(1, -1)
            close(got, want.numpy(), atol=2e-2, rtol=1e-2, what=f"dominant key at {far}, {pages} pages per wave")


@pytest.mark.parametrize("window", [70, 200, 1000])
@pytest.mark.parametrize("pages", [0, 1, 2, 8])
def test_attention_decode_window_edge(window, pages):
    """The lower edge of the window, to the key: a dominant key at position - window is out of
    the window and must count for nothing; at position - window + 1 it is the window's first key
    and must take all the weight.  On random data the keys before the edge are valid cache
    contents, and one key too many moves the output by less than the tolerance."""
    from sonicboom_amd import ops
    hq, hkv, hd, n = 6, 2, 64, 1500
    keys, vals, q, rise, scale = _looking_along_zero(n, hq, hkv, hd, 1, seed=41)
    table = torch.arange((n + 63) // 64, dtype=torch.int32).flip(0)[None, :].contiguous()
    group = hq // hkv
    for p in (n - 1, 1030, 1024 + window - 1):          # the edge inside a page, and on a page's first key
        p = min(p, n - 1)
        for inside in (False, True):
            k = keys.clone()
            edge = p - window + (1 if inside else 0)
            k[edge, :, 0] = rise
            kc, vc = fill_cache_from([k], [vals], table, BF16)
            pos = torch.tensor([p], dtype=torch.int32, device=DEV)
            with ops.attention_decode_pages_per_wave(hd, pages):
                got = ops.attention_decode_mfma(q.to(DEV), kc, vc, table.to(DEV), pos, hq, hkv, hd, scale, window)
            if inside:
                want = vals[edge].repeat_interleave(group, dim=0).reshape(1, -1).numpy()
            else:
                want = plain.attention(q.float().numpy(), k.reshape(n, -1).numpy(), vals.reshape(n, -1).numpy(), [p],
                                       np.arange(n), hq, hkv, hd, scale, causal=True, window=window)
                assert np.abs(want - vals[edge].repeat_interleave(group, dim=0).reshape(1, -1).numpy()).max() > 0.5
            close(got, want, atol=2e-2, rtol=1e-2, what=f"position {p}, window {window}, key {edge}")


@pytest.mark.parametrize("hq, hkv, hd", [(6, 2, 64), (28, 4, 128), (3, 1, 32)])
@pytest.mark.parametrize("window", [70, 300])
def test_attention_prefill_window_edge(hq, hkv, hd, window):
    """Prompt rows over a window: one dominant key at position d.  Rows up to d + window - 1
    have it as a key of their window (the last of them as its very first key) and must return
    its value; from row d + window on it has left the window and must count for nothing."""
    from sonicboom_amd import ops
    n = 700
    rows_pos = list(range(n - 80, n))
    keys, vals, q, rise, scale = _looking_along_zero(n, hq, hkv, hd, len(rows_pos), seed=51)
    group = hq // hkv
    table = torch.tensor([[7, 2, 9, 4, 0, 5, 1, 8, 3, 6, 10]], dtype=torch.int32)
    pos = torch.tensor(rows_pos, dtype=torch.int32)
    heights = (16, 32) if ops.attention_tall_ok(hq, hkv, hd) else (16,)
    # inside a tile of 16, at its end, at its start; at the end of a tile of 32, at its start
    for last_seeing in (rows_pos[0] + 20, rows_pos[0] + 47, rows_pos[0] + 48, rows_pos[0] + 63, rows_pos[0] + 64):
        d = last_seeing - window + 1
        k = keys.clone()
        k[d, :, 0] = rise
        kc, vc = fill_cache_from([k], [vals], table, BF16)
        want = plain.attention(q.float().numpy(), k.reshape(n, -1).numpy(), vals.reshape(n, -1).numpy(), rows_pos,
                               np.arange(n), hq, hkv, hd, scale, causal=True, window=window)
        v_d = vals[d].repeat_interleave(group, dim=0).reshape(1, -1).numpy()
        r = last_seeing - rows_pos[0]
        assert np.abs(want[r] - v_d).max() < 2e-2 and np.abs(want[r + 1] - v_d).max() > 0.5     # the case is sharp
        for height in heights:
            tiles = torch.tensor([(r0, min(height, len(rows_pos) - r0), 0, 0) for r0 in range(0, len(rows_pos), height)],
                                 dtype=torch.int32)
            got = ops.attention_prefill_mfma(q.to(DEV), kc, vc, table.to(DEV), pos.to(DEV), tiles.to(DEV), hq, hkv, hd,
                                             scale, window, tile_rows=height)
            close(got, want, atol=2e-2, rtol=1e-2, what=f"window {window}, dominant key {d}, tiles of {height}")


@pytest.mark.parametrize("hq, hkv, hd", [(4, 4, 16), (6, 2, 64), (2, 1, 96), (5, 1, 112), (28, 4, 128), (12, 2, 128)])
@pytest.mark.parametrize("window", [0, 70, 300])
@pytest.mark.parametrize("form", [1, 2])
def test_attention_prefill_forms(hq, hkv, hd, window, form):
    """Pages one by one through a block and pages cut over a block's waves, whichever the sizes would choose: whole
    prompts and a continuation in tiles of every height, and the edges of a window, up to six pages of which a block sees."""
    from sonicboom_amd import ops
    with ops.attention_prefill_form(form):
        test_attention_prefill_matrix_cores(hq, hkv, hd, min(window, 70))
        if window:
            test_attention_prefill_window_edge(hq, hkv, hd, window)


@pytest.mark.parametrize("hq, hkv, hd", [(4, 1, 64), (2, 1, 96), (5, 1, 112), (6, 2, 128)])
@pytest.mark.parametrize("window", [0, 577, 1000, 1024])
@pytest.mark.parametrize("missing", [(), (3, 10)])
def test_attention_prefill_waves_of_several_pages(hq, hkv, hd, window, missing):
    """Pages cut over a block's eight waves, ten to 28 of them, against 64 bits: waves with one, two and more pages, a window that starts
    in a wave's first page, on a page's first key and in the page after it, pages behind the window that are not in the table, keys that no
    row sees that are not numbers, and pages outside the cache as a wave's first and as a later one.  One key more or less at the
    window's edge, and every page, would show."""
    from sonicboom_amd import ops
    n, first = 1730, 1660                       # rows first .. n - 1
    rows = n - first
    width = -(-n // 64)
    lo_all = max(first - window + 1, 0) if window else 0
    table = torch.randperm(width + 3, generator=torch.Generator().manual_seed(5))[:width].to(torch.int32)[None, :]
    kc, vc = (randn(*shape, seed=2 + i).to(BF16) for i, shape in enumerate(((width + 3, hkv, 64, hd), (width + 3, hkv, hd, 64))))
    own = table[0].long()
    for p in range(lo_all - 1, lo_all + rows) if window else ():       # (large values where the rows' windows start)
        layout.put_value(vc, int(own[p // 64]), p % 64, 4.0 * layout.get_value(vc, int(own[p // 64]), p % 64).float())
    k = layout.keys_in_order(kc)[own].permute(0, 2, 1, 3).reshape(-1, hkv, hd)[:n]
    v = layout.values_in_order(vc)[own].permute(0, 3, 1, 2).reshape(-1, hkv, hd)[:n]
    none = torch.full((hkv, hd), float("nan"))
    for p in [*range(lo_all // 64 * 64, lo_all), *range(n, width * 64)]:
        layout.put_key(kc, int(table[0, p // 64]), p % 64, none)
        layout.put_value(vc, int(table[0, p // 64]), p % 64, none)
    first_page = lo_all // 64
    table[0, :first_page] = -1
    pos, key = torch.arange(first, n)[:, None], torch.arange(n)[None, :]
    seen = (key <= pos) & (key > pos - window if window else key >= 0)
    for i, page in enumerate(missing):
        table[0, first_page + page] = (-1, width + 3)[i]
        seen[:, (first_page + page) * 64:(first_page + page + 1) * 64] = False
    q = randn(rows, hq * hd, seed=7).to(BF16)
    views = q.view(rows, hq, hd)
    p, want, slack = attention_64(views, k, v, seen, hd ** -0.5)
    assert a_page_left_out_shows(p[:, :1], v, want[:1], slack[:1], hq)
    if window and not missing:
        for shift in (-1, 1):
            off = attention_64(views, k, v, (key <= pos) & (key > pos - window - shift), hd ** -0.5)[1]
            assert ((off - want).abs() > 2 * slack).any(2).any(1).all()
    for height in (16, 32) if ops.attention_tall_ok(hq, hkv, hd) else (16,):
        tiles = torch.tensor([(r, min(height, rows - r), 0, 0) for r in range(0, rows, height)], dtype=torch.int32)
        with ops.attention_prefill_form(2):
            got = ops.attention_prefill_mfma(q.to(DEV), kc.to(DEV), vc.to(DEV), table.to(DEV), pos[:, 0].to(torch.int32).to(DEV),
                                             tiles.to(DEV), hq, hkv, hd, hd ** -0.5, window, tile_rows=height)
        off = (got.cpu().double().view(rows, hq, hd) - want).abs()
        assert (off <= slack).all(), f"tiles of {height}: off by {off.nan_to_num(math.inf).max():.3g}"


@pytest.mark.parametrize("t, n, k", [(1, 4, 16), (3, 20, 40), (33, 100, 64), (70, 516, 1100), (40, 36, 2064)])
@pytest.mark.parametrize("out_dtype", [F32, BF16])
def test_float32_products_stored_by_fours(t, n, k, out_dtype):
    """Four neighbouring outputs at a time where rows start on 16 bytes, and one by one where they do not: the same bits, with a
    bias and a residual, in place, from packed and from row-major weights, and gated."""
    from sonicboom_amd import ops
    x, w, bias = randn(t, k).to(DEV), randn(n, k, seed=1).to(DEV), randn(n, seed=2).to(DEV)
    resid = randn(t, n, seed=3)
    off = torch.empty(t * n + 1, device=DEV)[1:].view(t, n)            # starts four bytes past sixteen
    off_out = torch.empty(t * n + 1, dtype=out_dtype, device=DEV)[1:].view(t, n)
    off.copy_(resid)
    packed = ops.pack_weight_f32(w)
    one = ops.gemm_f32(x, packed, bias, off, out_dtype, (n, k), out=off_out).clone()
    four = ops.gemm_f32(x, packed, bias, resid.to(DEV), out_dtype, (n, k))
    assert torch.equal(one, four)
    assert torch.equal(four, ops.gemm_plain(x, w, bias, resid.to(DEV), out_dtype))
    if out_dtype == F32:
        place = resid.to(DEV)
        assert torch.equal(ops.gemm_f32(x, packed, bias, place, F32, (n, k), out=place), four)
        want = x.cpu().double() @ w.cpu().double().T + bias.cpu().double() + resid.double()
        bound = (x.cpu().abs().double() @ w.cpu().abs().double().T + 4.0) * (k + 4) * 2.0 ** -24     # k roundings of the partial sums
        assert ((four.cpu().double() - want).abs() <= bound).all()
    h = n // 2
    pair = ops.pack_weight_f32(w, True)
    gated = ops.gemm_f32(x, pair, None, None, out_dtype, (n, k), gated="silu")
    off_gated = torch.empty(t * h + 1, dtype=out_dtype, device=DEV)[1:].view(t, h)
    assert torch.equal(gated, ops.gemm_f32(x, pair, None, None, out_dtype, (n, k), gated="silu", out=off_gated))


# (heads, head size, tile height, [(cached, rows)], window, whether the pages are cut over a block's waves); both forms measured
FORM_CHOICES = [
    (14, 2, 64, 16, [(0, 40)] * 16, 0, 0), (14, 2, 64, 16, [(0, 120)] * 8, 0, 0), (14, 2, 64, 16, [(200, 4)] * 64, 0, 0),
    (14, 2, 64, 16, [(0, 1000)], 0, 1), (14, 2, 64, 16, [(700, 300)], 0, 1), (14, 2, 64, 16, [(0, 16)] * 16, 0, 1),
    (14, 2, 64, 16, [(0, 33), (0, 255), (0, 700)], 0, 1), (16, 16, 64, 64, [(0, 40)] * 16, 0, 0), (16, 16, 64, 64, [(0, 1000)], 0, 1),
    (16, 16, 64, 64, [(0, 1000)], 100, 0), (4, 4, 64, 64, [(0, 60)] * 64, 0, 0), (16, 8, 64, 32, [(0, 10)] * 32, 0, 0),
    (32, 8, 96, 16, [(0, 16)] * 16, 0, 0), (32, 32, 128, 64, [(0, 130)], 0, 0), (12, 2, 128, 16, [(0, 10)] * 32, 0, 0),
    (12, 2, 128, 16, [(461, 61)] * 3, 0, 1), (28, 4, 128, 16, [(4000, 16)], 0, 1), (8, 1, 128, 16, [(1000, 16)] * 24, 0, 1),
    (28, 4, 128, 16, [(0, 1000)], 0, 0), (4, 2, 256, 16, [(4000, 16)], 0, 0)]


@pytest.mark.parametrize("hq, hkv, hd, height, seqs, window, keys", FORM_CHOICES)
def test_prefill_form_by_what_a_step_sees(hq, hkv, hd, height, seqs, window, keys):
    """Batches of short prompts keep the kernel that walks a tile's pages, which takes 0.6 to 0.9 of the other's time there."""
    from sonicboom_amd import ops
    from sonicboom_amd.engine.step import group_pages
    tiles = sum(-(-n // height) for _, n in seqs)
    groups = group_pages([n for _, n in seqs], [k for k, _ in seqs])
    lib = ops.library.attention_library(hd)
    assert lib.sb_attn_prefill_keys(tiles, height, hq, hkv, max(-(-(k + n) // 64) for k, n in seqs), window, *groups) == keys


@pytest.mark.parametrize("rows, width, n_in, inner", [(1, 16, 8, 16), (3, 104, 96, 40), (8, 896, 896, 200), (16, 72, 1032, 17), (5, 1536, 2048, 33)])
@pytest.mark.parametrize("gate", ["silu", "gelu_tanh", "relu"])
def test_products_that_carry_the_norm_between_them(rows, width, n_in, inner, gate):
    """The product that joins the stream and leaves an unfinished norm, and the gated one that finishes it, against 64 bits:
    one step of 32 k and less, waves without any, features and rows that fill no tile, with and without bias and weight."""
    from sonicboom_amd import ops
    x, w, b = randn(rows, n_in).to(BF16), randn(width, n_in, scale=0.1, seed=1).to(BF16), randn(width, seed=2)
    resid, nw = randn(rows, width, seed=3), randn(width, seed=4).to(BF16)
    wg = randn(2 * inner, width, scale=0.1, seed=5).to(BF16)
    for bias, weight in ((b, nw), (None, None)):
        want = resid.double() + x.double() @ w.double().T + (0.0 if bias is None else bias.double())
        stream = resid.to(DEV).clone()
        h = ops.gemm_split_join(x.to(DEV), ops.pack_weight(w.to(DEV)), None if bias is None else bias.to(DEV), stream,
                                None if weight is None else weight.to(DEV), 1e-6, packed_shape=(width, n_in))
        # float32 sums of n_in products of size 0.1: n_in 2^-24 of the sum of their magnitudes at most
        bound = (x.abs().double() @ w.abs().double().T + resid.abs().double() + 1.0) * (n_in + 4) * 2.0 ** -24
        assert ((stream.cpu().double() - want).abs() <= bound).all()
        now = stream.cpu().double()
        assert torch.allclose(h.ssq.cpu().double().sum(0), now.square().sum(1), rtol=1e-5)
        scaled = now * (1.0 if weight is None else weight.double())
        assert ((h.values.cpu().double() - scaled).abs() <= scaled.abs() * 2.0 ** -8 + 1e-30).all()
        got = ops.gemm_split_gated(h, ops.pack_weight(wg.to(DEV), True), gate, packed_shape=(2 * inner, width)).cpu().double()
        # from the same bfloat16 rows: float32 sums, then one rounding to bfloat16
        f = (now.square().mean(1, keepdim=True) + 1e-6).rsqrt()
        e = f * (h.values.cpu().double() @ wg.double().T)
        g, u = e[:, :inner], e[:, inner:]
        act = {"silu": torch.nn.functional.silu, "relu": torch.relu,
               "gelu_tanh": lambda v: torch.nn.functional.gelu(v, approximate="tanh")}[gate]
        ref = act(g) * u
        slack = (f * (h.values.cpu().double().abs() @ wg.double().abs().T)) * (width + 40) * 2.0 ** -24
        assert ((got - ref).abs() <= ref.abs() * 2.0 ** -8 + 1.2 * (slack[:, :inner] * u.abs() + slack[:, inner:] * g.abs()) + 1e-5).all()


# (rows, features, k): a tile of one feature, features and k that fill no tile, step or round, one block a tile and many, the most
# rows and the first that stay with the other kernels, X that just fits beside the sums in LDS and X that does not
ROWS_IN_LDS = [(1, 17, 512), (3, 40, 2560), (8, 264, 2568), (8, 4100, 1032), (5, 12300, 520), (8, 272, 7680), (8, 272, 7688), (9, 264, 1032),
               # as above where blocks that take a tile each stay behind: more than four rows of long products, long k
               (8, 13700, 2056), (5, 9000, 3200), (1, 40, 4104), (4, 264, 7680),
               # ... and where they do not: one slice of k to eight, a step a wave and remainders, many sums of squares a row
               (4, 13700, 2056), (8, 2064, 4096), (8, 2048, 4096), (2, 3000, 4088), (7, 9000, 904), (8, 1032, 1544),
               # X's share below 48 KB and past 64 KB with the block's own LDS, the most rows that this holds for, and the first past it
               (5, 264, 3584), (5, 272, 4096), (6, 264, 3584),
               # blocks of which a CU holds two, not three, and tiles for more than one round of either
               (8, 12304, 2560), (6, 12289, 2552)]


@pytest.mark.parametrize("rows, inner, width", ROWS_IN_LDS)
def test_gated_products_whose_blocks_keep_the_rows(rows, inner, width):
    """Against 64 bits, with an unfinished norm's factor; a row of infinities stays its own."""
    from sonicboom_amd import ops
    x, wg = randn(rows, width).to(BF16), randn(2 * inner, width, scale=0.1, seed=1).to(BF16)
    ssq = torch.rand((width + 15) // 16, rows, dtype=torch.float64, generator=torch.Generator().manual_seed(2)) * 16
    h = ops.ScaledRows(x.to(DEV), ssq.to(DEV), 1e-6)
    w = ops.pack_weight(wg.to(DEV), True)
    got = ops.gemm_split_gated(h, w, "relu", packed_shape=(2 * inner, width)).cpu().double()
    f = (ssq.sum(0) / width + 1e-6).rsqrt()[:, None]
    e, m = f * (x.double() @ wg.double().T), f * (x.double().abs() @ wg.double().abs().T) * (width + 40) * 2.0 ** -24
    g, u, mg, mu = torch.relu(e[:, :inner]), e[:, inner:], m[:, :inner], m[:, inner:]
    assert ((got - g * u).abs() <= (g * u).abs() * 2.0 ** -8 + 1.2 * (mg * u.abs() + mu * g)).all()
    if rows > 1:
        h.values[1, 3] = float("inf")
        again = ops.gemm_split_gated(h, w, "relu", packed_shape=(2 * inner, width)).cpu().double()
        rest = [i for i in range(rows) if i != 1]
        assert not torch.isfinite(again[1]).any()
        assert torch.equal(again[rest], got[rest])


@pytest.mark.parametrize("rows, n, k", [(1, 1000, 8184), (8, 8200, 520), (4, 2048, 2056), (8, 96, 61440), (8, 72, 70000), (9, 2048, 4096), (3, 20001, 136), (8, 17424, 7688),
                                        # one block a CU, and tiles that fill a round of one and not of two
                                        (8, 4112, 3584), (8, 8208, 4096)])
def test_raw_and_plain_products_whose_blocks_keep_the_rows(rows, n, k):
    """In K slices, and whole with float results where the matrix is wide, against 64 bits: cuts of K that the blocks' share of LDS
    allows and some that it does not."""
    from sonicboom_amd import ops
    x, w = randn(rows, k).to(BF16), randn(n, k, scale=0.1, seed=1).to(BF16)
    want, bound = x.double() @ w.double().T, (x.double().abs() @ w.double().abs().T) * (k + 8) * 2.0 ** -24
    packed = ops.pack_weight(w.to(DEV))
    part = ops.gemm_bf16_partial(x.to(DEV), packed, packed_shape=(n, k))
    assert ((part.cpu().double().sum(0) - want).abs() <= bound).all()
    whole = ops.gemm_bf16(x.to(DEV), packed, None, None, torch.float32, packed_shape=(n, k))
    assert ((whole.cpu().double() - want).abs() <= bound).all()


# (rows, features, k): 64- and 128-row tiles that make one round over the CUs, exactly and but for one, inner sizes of one to many
# stages, rows and features that end inside a tile, gated widths a little over a round, and the first that leave the rule
@pytest.mark.parametrize("rows, n, k", [(129, 2560, 2048), (400, 4608, 3584), (512, 4096, 64), (513, 4100, 192), (600, 4608, 640),
                                        (1300, 896, 896), (1301, 3072, 128), (183, 9728, 896), (183, 17920, 320)])
def test_tiled_products_of_one_round(rows, n, k):
    """The launcher's own choice, plain, gated and (where it cuts K) in slices, against 64 bits."""
    from sonicboom_amd import ops
    x, w = randn(rows, k).to(BF16), randn(n, k, scale=0.1, seed=1).to(BF16)
    want = (x.double() @ w.double().T)
    bound = (x.double().abs() @ w.double().abs().T) * (k + 8) * 2.0 ** -24
    packed = ops.pack_weight(w.to(DEV))
    got = ops.gemm_bf16(x.to(DEV), packed, None, None, F32, packed_shape=(n, k))
    assert ((got.cpu().double() - want).abs() <= bound).all()
    part = ops.gemm_bf16_partial(x.to(DEV), packed, packed_shape=(n, k))
    assert part is None or ((part.cpu().double().sum(0) - want).abs() <= bound).all()
    half = n // 2
    got = ops.gemm_bf16(x.to(DEV), ops.pack_weight(w.to(DEV), True), None, None, F32, gated="relu", packed_shape=(n, k)).cpu().double()
    g, u, mg, mu = torch.relu(want[:, :half]), want[:, half:], bound[:, :half], bound[:, half:]
    assert ((got - g * u).abs() <= (g * u).abs() * 2.0 ** -22 + 1.1 * (mg * u.abs() + mu * g) + mg * mu).all()


# (width, groups, offset): lengths that a wave's four registers of four just hold and just do not, parts that no four divides, a row
# off 16 bytes, groups that leave waves idle, more groups than waves
@pytest.mark.parametrize("width, groups, offset", [(4096, 2, 0), (4104, 2, 0), (4096, 4, 0), (4112, 4, 0), (2048, 2, 4), (3072, 3, 0), (3084, 3, 0), (4095, 5, 0),
                                                   (4100, 5, 0), (60, 5, 0), (64, 16, 0), (8, 2, 0), (90, 9, 0)])
@pytest.mark.parametrize("out_dtype, w_dtype", [(F32, F32), (BF16, BF16), (F32, None)])
def test_norms_in_groups(width, groups, offset, out_dtype, w_dtype):
    """Against 64 bits: a sum in double, and four float roundings behind it (the factor's two, by the row, by the weight)."""
    from sonicboom_amd import ops
    rows = 5
    w = None if w_dtype is None else (1.0 + randn(width, scale=0.1)).to(w_dtype)
    x = torch.empty(rows * width + 4, device=DEV)[offset // 4:][:rows * width].view(rows, width).copy_(randn(rows, width, scale=3.0))
    pick = torch.tensor([4, 0, 4], dtype=torch.int32, device=DEV)
    f = x.cpu().double().view(rows, groups, -1)
    want = (f / (f.square().mean(-1, keepdim=True) + 1e-6).sqrt()).view(rows, width) * (1.0 if w is None else w.double())
    for index in (None, pick):
        got = ops.rmsnorm(x, None if w is None else w.to(DEV), 1e-6, out_dtype, index, groups).cpu().double()
        ref = want if index is None else want[index.cpu().long()]
        assert ((got - ref).abs() <= ref.abs() * (2.0 ** -21 + (2.0 ** -8 if out_dtype == BF16 else 0.0))).all()


# sequences of less than four rows and of remainders, of one chunk, of eight, of more than eight and of none of their own
def test_gated_recurrence_in_chunks_of_every_remainder():
    """In chunks against the walk of the same kernel's rows: the states meet through products of at most one, so both are within the
    roundings of a sum as long as the sequence."""
    from sonicboom_amd import ops
    from sonicboom_amd.engine.step import row_runs
    step = ops.mingru_chunk_rows()
    lengths, width = [1, 3, 4, 5, step - 1, step, step + 1, 7 * step, 8 * step, 8 * step + 2, 9 * step - 3, 2], 70
    cu = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    slots = np.arange(len(lengths), dtype=np.int32)[::-1].copy()
    p, state = randn(int(cu[-1]), 3 * width, scale=2.0).to(DEV), randn(len(lengths), width, seed=1).to(DEV)
    dev = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.int32).to(DEV)
    walked, chunked = state.clone(), state.clone()
    want = ops.mingru_scan(p, walked, dev(cu), dev(slots), len(lengths), F32)
    got = ops.mingru_scan(p, chunked, dev(cu), dev(slots), len(lengths), F32, dev(row_runs(lengths, cu, step)))
    # |state| stays below the largest start or candidate, about 10: some hundred rows' roundings of 2^-24 of that, decayed
    close(chunked, walked.cpu(), atol=1e-5, rtol=1e-5, what="states")
    close(got, want.cpu(), atol=1e-5, rtol=1e-5, what="rows")


def test_the_norm_between_two_products_sums_in_double():
    """Rows whose squares are float numbers but whose sum of squares over the width is none, and rows of many small numbers
    beside a large one: the factor follows from the sum in double, as of every RMS norm."""
    from sonicboom_amd import ops
    rows, width, n_in, inner = 4, 3584, 64, 48
    x, w = torch.zeros(rows, n_in, dtype=BF16).to(DEV), randn(width, n_in, seed=1).to(BF16).to(DEV)
    resid = randn(rows, width, seed=2)
    resid[0] = 1.5e19 * torch.sign(resid[0])               # 2.25e38 each, 8.1e41 in all
    resid[1, 0], resid[1, 1:] = 3e4, 1.0                   # every square of 1 lies below half a unit of the last place of 9e8
    resid[2] *= 1e-18
    wg = randn(2 * inner, width, scale=0.1, seed=5).to(BF16)
    h = ops.gemm_split_join(x, ops.pack_weight(w), None, resid.to(DEV), None, 1e-6, packed_shape=(width, n_in))
    squares = (resid * resid).double().sum(1)
    # sums of 3,584 squares in double: exact to 2^-40
    assert h.ssq.dtype == torch.float64 and ((h.ssq.cpu().sum(0) - squares).abs() <= squares * 2.0 ** -40).all()
    got = ops.gemm_split_gated(h, ops.pack_weight(wg.to(DEV), True), "relu", packed_shape=(2 * inner, width)).cpu().double()
    f = (squares / width + 1e-6).rsqrt()[:, None]
    e = f * (h.values.cpu().double() @ wg.double().T)
    slack = (f * (h.values.cpu().double().abs() @ wg.double().abs().T)) * (width + 40) * 2.0 ** -24
    g, u, sg, su = e[:, :inner], e[:, inner:], slack[:, :inner], slack[:, inner:]
    assert torch.isfinite(got).all() and got[0].abs().max() > 0.1
    assert ((got - torch.relu(g) * u).abs() <= (torch.relu(g) * u).abs() * 2.0 ** -8 + 1.2 * (sg * u.abs() + su * g.abs()) + 1e-5).all()


@pytest.mark.parametrize("width, heads, inner, rows", [(128, 2, 320, 9), (5120, 40, 320, 1), (8192, 64, 320, 4), (8192, 64, 320, 5),
                                                        (3072, 24, 8960, 2)])
def test_decode_steps_on_both_sides_of_the_rule_for_the_norm(width, heads, inner, rows):
    """The norm rides in the products, or is a pass between them: the same logits but for the order of a norm's factor and of
    sums, and the rule asks for what the sizes take."""
    from sonicboom_amd import ops
    from sonicboom_amd.engine import DecoderModel, Engine, StepEntry
    from sonicboom_amd.ops import kernels
    cfg = {"architectures": ["Qwen2ForCausalLM"], "num_hidden_layers": 2, "hidden_size": width, "num_attention_heads": heads,
           "num_key_value_heads": 1, "intermediate_size": inner, "vocab_size": 300, "rope_theta": 10000.0, "rms_norm_eps": 1e-6,
           "max_position_embeddings": 256, "tie_word_embeddings": True}
    model = DecoderModel.from_random(cfg, 3, "bfloat16", DEV)
    eng = Engine(model, 64 * rows, max_slots=rows)
    joined = []
    real = kernels.gemm_split_join
    rides = ops.split_norm_pays(rows, width, inner)
    assert rides == (rows <= 8 and (width <= 4096 or (width == 8192 and rows <= 4)))
    out = []
    for most in (kernels.SPLIT_MAX_ROWS, 0):
        with pytest.MonkeyPatch.context() as mp:
            mp.setattr(ops, "gemm_split_join", lambda *a, **k: (joined.append(most), real(*a, **k))[1])
            mp.setattr(kernels, "SPLIT_MAX_ROWS", most)
            slots = [eng.alloc_slot() for _ in range(rows)]
            eng.step([StepEntry(s, [5 + i, 7], ()) for i, s in enumerate(slots)])
            out.append(eng.step([StepEntry(s, [11 + i], (0,)) for i, s in enumerate(slots)]).float().cpu())
            for s in slots:
                eng.free_slot(s)
    assert joined == ([kernels.SPLIT_MAX_ROWS] * 2 if rides else [])
    # a rounding of the normed rows to bfloat16 (2^-9) at another place in each of two layers
    assert (out[0] - out[1]).abs().max() <= 0.05 * out[0].std()


def test_projections_of_rows_off_sixteen_bytes():
    """Rows that start between two 16-byte lines: whole, gated, and joined to the stream with a norm to follow, where the
    product that carries the norm stands back."""
    from types import SimpleNamespace
    from sonicboom_amd import ops
    from sonicboom_amd.parts.linear import Linear
    rows, n_in, width = 3, 96, 104
    x, w = randn(rows, n_in).to(BF16).to(DEV), randn(width, n_in, scale=0.1, seed=1).to(BF16).to(DEV)
    off = torch.empty(rows * n_in + 4, dtype=BF16, device=DEV)[4:].view(rows, n_in).copy_(x)
    assert off.data_ptr() % 16 == 8
    norm = SimpleNamespace(fusable=True, groups=1, weight=None, eps=1e-6)
    lin = Linear(w, None)
    assert lin.joins(x, norm) and not lin.joins(off, norm)
    for rows_ in (x, off):
        resid = torch.ones(rows, width, device=DEV)
        lin.add_into(rows_, resid, norm, BF16)
        close(resid, ref_gemm(x.cpu(), w.cpu()) + 1.0, atol=1e-4, rtol=1e-5, what="joined")
    gated = Linear(w, None, gated=True)
    assert torch.equal(gated(off, F32), gated(x, F32)) and torch.equal(lin(off, F32), lin(x, F32))


FOLDED_SHAPES = [(4, 2, 16, 16), (3, 1, 32, 32), (5, 5, 48, 16), (6, 2, 80, 64), (28, 4, 128, 128), (16, 1, 64, 0),
                 (2, 1, 256, 256)]


def folded_against_two_kernels(hq, hkv, hd, rot, window, pages, lens, alike=False):
    from sonicboom_amd import ops
    n_seq = len(lens)
    width_pages = max((n + 63) // 64 for n in lens)
    perm = torch.randperm(n_seq * width_pages + 3, generator=torch.Generator().manual_seed(5))
    table = torch.full((n_seq, width_pages), -1, dtype=torch.int32)
    it = iter(perm.tolist())
    for s_, n in enumerate(lens[:-1]):            # the last sequence keeps a table of -1
        for pg in range((n + 63) // 64):
            table[s_, pg] = next(it)
    n_pages = n_seq * width_pages + 3
    kc0 = randn(n_pages, hkv, 64, hd, seed=1).to(BF16)
    vc0 = randn(n_pages, hkv, hd, 64, seed=2).to(BF16)
    pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32)
    pos[-1] = 0
    seq = torch.arange(n_seq, dtype=torch.int32)
    width = (hq + 2 * hkv) * hd
    inv = ff = None
    if rot:
        inv = torch.exp(-2.0 * torch.arange(rot // 2, dtype=F32) / rot * math.log(1e4)).to(DEV)
        ff = (1.0 + torch.arange(rot // 2, dtype=F32) / rot).to(DEV)
    scale = 1.0 / math.sqrt(hd)
    for n_slices in (1, 3):
        qkv = randn(n_slices, n_seq, width, seed=3 + n_slices).to(DEV)
        bias = randn(width, seed=9, scale=0.3).to(DEV) if n_slices > 1 else None
        arg = qkv if n_slices > 1 else qkv[0].contiguous()
        # two kernels
        kc1, vc1 = kc0.clone().to(DEV), vc0.clone().to(DEV)
        q = ops.rope_kv_store(arg, BF16, inv, ff, rot, pos.to(DEV), seq.to(DEV), kc1, vc1, table.to(DEV), hq, hkv, hd,
                              bias=bias)
        with ops.attention_decode_pages_per_wave(hd, pages):
            want = ops.attention_decode_mfma(q, kc1, vc1, table.to(DEV), pos.to(DEV), hq, hkv, hd, scale, window, alike=alike)
            # one kernel
            kc2, vc2 = kc0.clone().to(DEV), vc0.clone().to(DEV)
            assert ops.attention_decode_rope_ok(arg, BF16, BF16, hq, hkv, hd, rot)
            got = ops.attention_decode_rope(arg, inv, ff, rot, kc2, vc2, table.to(DEV), pos.to(DEV), hq, hkv, hd, scale,
                                            window, bias=bias, alike=alike)
            assert torch.equal(got.view(torch.int16), want.view(torch.int16)), f"slices {n_slices}"
            assert torch.equal(kc2.view(torch.int16), kc1.view(torch.int16))
            assert torch.equal(vc2.view(torch.int16), vc1.view(torch.int16))
            assert not torch.equal(kc2.view(torch.int16), kc0.to(DEV).view(torch.int16))     # something was stored
            # queries only (a layer that reads another layer's cache): nothing is stored
            kc3, vc3 = kc1.clone(), vc1.clone()
            only_q = arg[..., : hq * hd].contiguous()
            got = ops.attention_decode_rope(only_q, inv, ff, rot, kc3, vc3, table.to(DEV), pos.to(DEV), hq, hkv, hd,
                                            scale, window, bias=bias, store=False, alike=alike)
            assert torch.equal(got.view(torch.int16), want.view(torch.int16))
            assert torch.equal(kc3.view(torch.int16), kc1.view(torch.int16))
    assert not ops.attention_decode_rope_ok(arg, BF16, BF16, 34, 2, hd, rot)          # 17 heads per kv head


@pytest.mark.parametrize("hq, hkv, hd, rot, pages", [(*sh, p) for sh in FOLDED_SHAPES for p in (0, 1, 2, 8)
                                                     if p <= 1 or sh[2] <= 128])     # several pages per wave: up to head size 128
@pytest.mark.parametrize("window", [0, 70])
def test_attention_decode_with_rotation_and_store_folded_in(hq, hkv, hd, rot, window, pages):
    """A decode step's rotation, store and attention in one kernel against the two kernels one
    after the other: the same output and the same cache, bit for bit.  The qkv rows come as one
    array and as three K slices with a bias; rows stand at a page's first and last slot, on the
    first token of a sequence, and behind a window; one row has no page at all (a row added to
    fill a batch: nothing is stored, nothing seen)."""
    folded_against_two_kernels(hq, hkv, hd, rot, window, pages, [1, 64, 65, 128, 300, 700, 1])


@pytest.mark.parametrize("hq, hkv, hd, rot", FOLDED_SHAPES)
@pytest.mark.parametrize("window", [0, 70])
@pytest.mark.parametrize("lens", [[1, 64, 256, 257, 320, 1], [100, 150, 350, 1], [400, 1], [1, 257, 320, 321, 384, 385, 448, 449, 512, 1]],
                         ids=lambda n: f"to{max(n)}")
def test_attention_decode_folded_in_where_one_block_takes_a_row(hq, hkv, hd, rot, window, lens):
    """The same where a table has five to eight pages and eight waves take a row (heads of up to 128 numbers): the row's own
    page with each of the eight waves, at its first and last slots and inside."""
    folded_against_two_kernels(hq, hkv, hd, rot, window, 0, lens)


# (heads, kv heads, head size, the rows' numbers of keys): rows past the 64 that a wave looks at at once, two tiles of heads a kv head, a
# wave's share of one page and of several, rows that stay whole, one long row among short ones; and tables short beside the rows, which come
# in equal chunks whatever their lengths: one page a row, rows in one chunk and in more
DEALT = [(4, 2, 16, [1 + 31 * i % 2100 for i in range(130)]), (20, 1, 64, [64 * (1 + 7 * i % 23) for i in range(70)]),
         (28, 4, 32, [2000 + 97 * i for i in range(33)]), (28, 4, 128, [640 - i % 3 for i in range(64)]), (14, 2, 64, [20000] + [5] * 40),
         (8, 8, 48, [30 + i for i in range(33)]), (4, 2, 16, [1 + 31 * i % 5000 for i in range(130)]), (4, 4, 64, [1950 - i % 3 for i in range(64)]),
         (7, 1, 128, [1 + 61 * i % 1000 for i in range(150)])]


def attention_64(q, k, v, seen, scale):
    """Rows q [n, heads, d] over keys k and values v [m, kv heads, d] in 64 bits, `seen` bool [n, m]: the weights [heads, n, m], the results
    [n, heads, d], and how far a kernel may be off them.  It rounds every weight to bfloat16, by up to 2^-9 of it and so by 0.58 of that
    in the root mean square: 2^-7 sqrt(sum p^2 v^2) is seven times what these roundings add up to.  The result is rounded once more."""
    group = q.shape[1] // k.shape[1]
    k, v = (t.double().repeat_interleave(group, 1).transpose(0, 1) for t in (k, v))
    s = q.double().transpose(0, 1) @ k.transpose(1, 2) * scale
    p = torch.softmax(s.masked_fill(~seen, -math.inf), -1).nan_to_num(0.0)
    out, spread = p @ v, ((p * p) @ (v * v)).sqrt()
    return p, out.transpose(0, 1), (2.0 ** -7 * spread + 2.0 ** -8 * out.abs() + 1e-6).transpose(0, 1)


def a_page_left_out_shows(p, v, out, slack, hq):
    """Whether every page of which a row (n = 1) sees half or more would be missed: results without it lie outside of what two kernels within
    the slack can differ by."""
    v = v.double().repeat_interleave(hq // v.shape[1], 1)
    for lo in range(0, p.shape[2], 64):
        w = p[:, :, lo:lo + 64]
        if int((w[0] > 0).sum()) < 32 or float(w.sum(-1).max()) > 1 - 1e-9:
            continue
        without = (out - (w @ v[lo:lo + 64].transpose(0, 1)).transpose(0, 1)) / (1 - w.sum(-1)).T[:, :, None]
        if not ((without - out).abs() > 2 * slack).any():
            return False
    return True


@pytest.mark.parametrize("hq, hkv, hd, lens", DEALT, ids=lambda v: f"{len(v)}rows" if isinstance(v, list) else str(v))
@pytest.mark.parametrize("window", [0, 70, 1000])
def test_attention_decode_deals_pages_out(hq, hkv, hd, lens, window):
    """Many rows of unequal length, whose pages the kernel deals out to its blocks or, told that they are alike, cuts into as many chunks
    each: against 64 bits, and against blocks of four pages of a row each, the same sums of float32 numbers in another order, then one
    rounding to bfloat16.  Every ninth row has no page."""
    from sonicboom_amd import ops
    width = max(-(-n // 64) for n in lens)
    assert -(-width // 8) * len(lens) * hkv * -(-(hq // hkv) // 16) >= 256
    table = torch.full((len(lens), width), -1, dtype=torch.int32)
    n_pages = sum(-(-n // 64) for n in lens) + 3
    pages = iter(torch.randperm(n_pages, generator=torch.Generator().manual_seed(1)).tolist())
    for i, n in enumerate(lens):
        for pg in range(-(-n // 64)):
            table[i, pg] = next(pages)
        if window:
            table[i, :max(n - window, 0) // 64] = -1         # the cache gives pages behind a window back
        if i % 9 == 5:
            table[i] = -1
    kc, vc = (randn(*shape, seed=2).to(BF16).to(DEV) for shape in ((n_pages, hkv, 64, hd), (n_pages, hkv, hd, 64)))
    q, pos = randn(len(lens), hq * hd, seed=3).to(BF16).to(DEV), torch.tensor([n - 1 for n in lens], dtype=torch.int32).to(DEV)
    run = lambda **how: ops.attention_decode_mfma(q, kc, vc, table.to(DEV), pos, hq, hkv, hd, hd ** -0.5, window, **how).float()
    got, again = run(), run()
    with ops.attention_decode_pages_per_wave(hd, 1):
        want = run()
    assert torch.equal(got, again)
    assert (got[5::9] == 0).all() and want.abs().max() > 0.1
    # probabilities are rounded to bfloat16 (2^-9 of each) relative to another maximum, as keys meet in other steps: the sums' part
    # in that is at most 2^-8 of the values' largest, and half of one rounding of each result
    assert ((got - want).abs() <= 2.0 ** -8 * vc.float().abs().max() * 0.5 + want.abs() * 2.0 ** -8).all()
    alike = run(alike=True)
    if not ops.attention_decode_alike_pays(len(lens), hq, hkv, hd, width):       # (a short table: the word is not heard)
        assert width * (hd + 64) <= 12 * (len(lens) * hkv * -(-(hq // hkv) // 16) + 64) and torch.equal(alike, got)
    k_all, v_all = layout.keys_in_order(kc.cpu()), layout.values_in_order(vc.cpu())
    longest = max((i for i in range(len(lens)) if i % 9 != 5), key=lambda i: lens[i])
    for i, n in enumerate(lens):
        if i % 9 == 5:
            assert (alike[i] == 0).all()
            continue
        own = table[i, :-(-n // 64)].long().clamp(min=0)     # (pages behind the window: whatever is there, not seen)
        k = k_all[own].permute(0, 2, 1, 3).reshape(-1, hkv, hd)[:n]
        v = v_all[own].permute(0, 3, 1, 2).reshape(-1, hkv, hd)[:n]
        seen = (torch.arange(n) > n - 1 - window) if window else torch.ones(n, dtype=torch.bool)
        p, ref, slack = attention_64(q[i:i + 1].cpu().view(1, hq, hd), k, v, seen[None, :], hd ** -0.5)
        for name, out in (("dealt out", got), ("alike", alike)):
            off = (out[i].cpu().double().view(1, hq, hd) - ref).abs()
            assert (off <= slack).all(), f"{name}, row {i} of {n} keys: off by {off.max():.3g}, {(off / slack).max():.3g} of the slack"
        if i == longest:
            assert a_page_left_out_shows(p, v, ref, slack, hq)


# (heads, kv heads, head size, rotary width): more rows than a wave looks at at once, of lengths from one key on
@pytest.mark.parametrize("hq, hkv, hd, rot, lens", [(14, 2, 64, 64, [1 + 37 * i % 1500 for i in range(130)]), (28, 4, 128, 128, [60 + 131 * i % 1400 for i in range(70)]),
                                                    (16, 1, 128, 64, [30 + 211 * i % 6000 for i in range(65)]), (8, 8, 80, 0, [64 * (1 + 5 * i % 40) for i in range(20)]),
                                                    (14, 2, 64, 64, [1 + 37 * i % 2400 for i in range(130)]), (28, 4, 128, 128, [1 + 97 * i % 500 for i in range(40)])],
                         ids=lambda v: f"{len(v)}rows" if isinstance(v, list) else str(v))
@pytest.mark.parametrize("window, alike", [(0, False), (0, True), (300, False), (300, True)])
def test_attention_decode_folded_in_where_pages_are_dealt_out(hq, hkv, hd, rot, lens, window, alike):
    assert -(-max(lens) // 64 // 8) * len(lens) * hkv >= 256 or (len(lens) * hkv > 128 and max(lens) > 4 * 64)
    folded_against_two_kernels(hq, hkv, hd, rot, window, 0, lens, alike)


def test_attention_decode_of_like_rows_needs_no_second_kernel():
    """Where rows of like length fill the GPU by themselves every row is one chunk, and chunks a row grow as rows get fewer."""
    from sonicboom_amd.ops import library
    cut = library.attention_library(128).sb_attn_decode_cut
    assert [cut(n, 28, 4, 48) for n in (48, 64, 128)] == [1, 1, 1]
    assert 1 < cut(16, 28, 4, 80) <= cut(8, 28, 4, 144) <= 16
    assert cut(2, 28, 4, 512) == 0 and cut(64, 28, 4, 4) == 0 and cut(64, 28, 4, 20) == 0 and cut(8, 28, 4, 8) == 0
    # (few rows, and tables short beside the rows: the word is not heard)
    assert library.attention_library(256).sb_attn_decode_cut(64, 28, 4, 48) == 0


@pytest.mark.parametrize("vocab", [5, 256, 1000, 152064])
def test_argmax_first_maximum(vocab):
    from sonicboom_amd import ops
    x = randn(6, vocab)
    x[0, :] = 0.5                                   # all equal: id 0
    x[1, vocab - 1] = 50.0
    x[2, 3] = 60.0
    if vocab > 4:
        x[2, 4] = 60.0                              # a tie: the lower id
    x[3, :] = float("-inf")
    got = ops.argmax(x.to(DEV)).cpu().tolist()
    want = [plain.argmax(r.numpy()) for r in x]
    assert got == want and got[:3] == [0, vocab - 1, 3]


@pytest.mark.parametrize("vocab", [7, 256, 300, 5000, 8192, 8193, 12289, 152064])
@pytest.mark.parametrize("temperature", [1.0, 0.7])
def test_top_candidates(vocab, temperature):
    """Rows short enough for one block, and rows cut into parts of 4,096 whose best are merged
    (from 8,193 on; a last part of one element; a part that holds all of the best)."""
    from sonicboom_amd import ops
    x = randn(6, vocab, scale=2.0)
    x[1] = torch.round(x[1])                        # many ties: ordered by id
    x[2, :] = 1.25                                  # all equal
    x[3, ::3] = -0.0
    x[3, 1::3] = 0.0                                # signed zeros are one value
    x[4, vocab // 3:] = -float("inf")               # fewer finite values than candidates, perhaps
    x[5, -min(300, vocab):] += 50.0                 # all of the best at the row's end
    k = min(256, vocab)
    ids, z = ops.top_candidates(x.to(DEV), temperature, k)
    ids, z = ids.cpu().numpy(), z.cpu().numpy()
    for r in range(6):
        want = sampling_plain.select_candidates(x[r].numpy(), temperature)
        assert [c[0] for c in want] == ids[r].tolist(), f"row {r}"
        assert np.array_equal(np.array([c[1] for c in want], dtype=np.float32), z[r]), f"row {r}"


@pytest.mark.parametrize("params", [
    dict(temperature=0.8), dict(temperature=1.3, top_k=5), dict(temperature=0.5, top_p=0.7),
    dict(temperature=1.0, min_p=0.2), dict(temperature=0.9, top_k=40, top_p=0.9, min_p=0.01),
    dict(temperature=0.05, top_p=0.5), dict(temperature=2.0, top_k=1), dict(temperature=1.0, top_p=1e-9, min_p=1.0),
    dict(temperature=1.0, top_k=300, top_p=0.999),
])
@pytest.mark.parametrize("vocab", [40, 400, 5000])
def test_draw_equals_the_plain_sampler(params, vocab):
    """Filters and Gumbel draw on the device, a wave a row: every row gets the token that the
    plain sampler draws for it alone (flat and peaked rows, ties among the best, one candidate far
    above the window, positions past 2^32, a 64-bit seed, fewer logits than candidates)."""
    from sonicboom_amd import ops
    SP = sampling_plain
    r = np.random.default_rng(vocab)
    rows = []
    for i in range(96):
        logits = (r.standard_normal(vocab) * (0.2 if i % 5 == 0 else 3.0)).astype(np.float32)
        if i % 7 == 3:
            logits[10:20] = logits[5]
        if i % 6 == 1:
            logits[3] = 80.0
        rows.append(logits)
    positions = [int(q) for q in r.integers(0, 5000, size=len(rows))]
    positions[0], positions[1] = 0, 2 ** 33 + 5
    seed = 0x9E3779B97F4A7C15
    t = params["temperature"]
    k = min(ops.MAX_CANDIDATES, vocab)
    ids, z = ops.top_candidates(torch.tensor(np.stack(rows), device=DEV), t, k)
    log_min_p = float(np.log(np.float32(params["min_p"]))) if params.get("min_p", 0.0) > 0.0 else None
    top_p = float(np.float64(np.float32(params["top_p"]))) if 0.0 < params.get("top_p", 1.0) < 1.0 else None
    got = ops.draw(ids, z, positions, params.get("top_k", 0), log_min_p, top_p, seed).tolist()
    for i, logits in enumerate(rows):
        kept = SP.filter_candidates(SP.select_candidates(logits, t), params.get("top_k", 0),
                                    params.get("top_p", 1.0), params.get("min_p", 0.0))
        assert got[i] == SP.draw(kept, seed, positions[i]), f"row {i}"


def test_draw_at_the_positions_after_device_side_lengths():
    """Lengths as a decode step keeps them on the device (int32): the new token's position is
    length + 1, and the tokens are those of the same positions brought from the host."""
    from sonicboom_amd import ops
    r = np.random.default_rng(3)
    logits = torch.tensor((r.standard_normal((40, 3000)) * 2.0).astype(np.float32), device=DEV)
    ids, z = ops.top_candidates(logits, 0.9, ops.MAX_CANDIDATES)
    lengths = [int(q) for q in r.integers(0, 4000, size=40)]
    want = ops.draw(ids, z, [n + 1 for n in lengths], 50, None, 0.9, 12345).tolist()
    out = torch.full((40,), -7, dtype=torch.int32, device=DEV)
    got = ops.draw(ids, z, torch.tensor(lengths, dtype=torch.int32, device=DEV), 50, None, 0.9, 12345, out=out)
    assert got is out and out.tolist() == want
    assert ops.draw(ids, z, lengths, 50, None, 0.9, 12345).tolist() != want       # other positions, other draws


def test_draw_keeps_no_candidate_of_an_empty_row():
    """A row whose candidates all lie outside (ids of -1, as a row shorter than k is filled)
    gives -1; its neighbours are not disturbed."""
    from sonicboom_amd import ops
    ids = torch.tensor([[3, 1, -1, -1], [-1, -1, -1, -1]], dtype=torch.int32, device=DEV)
    z = torch.tensor([[2.0, 1.0, 0.0, 0.0], [0.0, 0.0, 0.0, 0.0]], dtype=torch.float32, device=DEV)
    got = ops.draw(ids, z, [5, 6], 0, None, None, 1).tolist()
    assert got[0] in (3, 1) and got[1] == -1


@pytest.mark.parametrize("exact", [False, True])
def test_penalize(exact):
    from sonicboom_amd import ops
    logits = randn(3, 50)
    hist = [[1, 2, 2, 49], [], [7] * 10]
    rows, toks, counts = [0, 0, 0, 2], [1, 2, 49, 7], [1, 2, 1, 10]
    dev = logits.to(DEV)
    ops.penalize(dev, *(torch.tensor(v, dtype=torch.int32, device=DEV) for v in (rows, toks, counts)),
                 1.3, 0.2, 0.1, exact)
    for r in range(3):
        want = sampling_plain.penalize(logits[r].numpy(), exact, 1.3, 64, 0.2, 0.1, hist[r])
        assert np.array_equal(dev[r].cpu().numpy(), want), f"row {r}"

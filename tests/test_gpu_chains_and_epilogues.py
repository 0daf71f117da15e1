"""Float32 products in their chains, gated products whose weights pass through registers, xIELU as a pass and on a product's way out."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F32, BF16 = "cuda:0", torch.float32, torch.bfloat16


def randn(*shape, seed=0, scale=1.0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale


@pytest.mark.parametrize("t", [1, 16, 20, 70])
@pytest.mark.parametrize("n, k", [(40, 256), (40, 260), (33, 768), (33, 1024), (48, 1280), (16, 2304)])
def test_float32_chains_end_inside_and_between_segments(t, n, k):
    """One to four chains of 256 k, two and three of 1,024: the same bits from every kernel, within a chain's roundings of 64 bits."""
    from sonicboom_amd import ops
    x, w = randn(t, k, seed=t), randn(n, k, seed=k, scale=0.05)
    want = ops.gemm_plain(x.to(DEV), w.to(DEV), None, None, F32)
    got = ops.gemm_f32(x.to(DEV), ops.pack_weight_f32(w.to(DEV)), None, None, F32, (n, k))
    assert torch.equal(got, want)
    # each of at most a chain's and four more roundings is half a unit of a running sum that the terms' absolute values bound
    bound = ((1024 if k > 1024 else 256) + 4) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert ((got.cpu().double() - x.double() @ w.double().T).abs() <= bound).all()
    if n % 2 == 0:
        gated = ops.gemm_f32(x.to(DEV), ops.pack_weight_f32(w.to(DEV), True), None, None, F32, (n, k), gated="silu")
        assert torch.equal(gated, ops.silu_mul(want, F32))


@pytest.mark.parametrize("t, n, k", [(515, 3001, 901), (515, 3001, 1029), (4033, 700, 272), (129, 9000, 2300)])
def test_row_major_products_of_many_tiles_have_the_bits_of_packed_ones(t, n, k):
    """Rows, columns and k that end inside a tile and a stage, one chain to four, two and three of 1,024."""
    from sonicboom_amd import ops
    for dtype in (F32, BF16):
        x, w = randn(t, k, seed=t).to(DEV, dtype), randn(n, k, seed=k, scale=0.05).to(DEV, dtype)
        want = ops.gemm_f32(x.float(), ops.pack_weight_f32(w.float()), None, None, F32, (n, k))
        assert torch.equal(ops.gemm_plain(x, w, None, None, F32), want)


@pytest.mark.parametrize("shape", [6, 7, 8])
@pytest.mark.parametrize("t, inner, k", [(65, 64, 64), (96, 72, 320), (97, 132, 384), (129, 20, 448), (193, 260, 896), (400, 64, 192)])
def test_gated_products_with_weights_through_registers(shape, t, inner, k):
    """Rows and columns that end inside a tile, stage counts on either side of the ring of six."""
    from sonicboom_amd import ops
    x, w = randn(t, k, seed=t).to(BF16), randn(2 * inner, k, seed=k, scale=0.05).to(BF16)
    gu = x.double() @ w.double().T
    g, u = gu[:, :inner], gu[:, inner:]
    packed = ops.pack_weight(w.to(DEV), True)
    for act, want in (("silu", g / (1.0 + torch.exp(-g)) * u), ("relu", torch.relu(g) * u),
                      ("gelu_tanh", 0.5 * g * (1 + torch.tanh(0.7978845608028654 * g * (1 + 0.044715 * g * g))) * u)):
        with ops.gemm_tile_shape(shape, "direct"):
            got = ops.gemm_bf16(x.to(DEV), packed, None, None, F32, gated=act, packed_shape=(2 * inner, k))
            half = ops.gemm_bf16(x.to(DEV), packed, None, None, BF16, gated=act, packed_shape=(2 * inner, k))
        assert ((got.cpu().double() - want).abs() <= 1e-4 * math.sqrt(k) + 1e-4 * want.abs()).all(), act
        assert torch.equal(half, got.to(BF16)), act


@pytest.mark.parametrize("inner, rows", [(1024, (1024, 1536, 2048, 3072)), (64, (16384,)), (11008, (65, 96))])
def test_gated_products_on_either_side_of_a_round_of_tiles(inner, rows):
    """The launcher's own choice where 64, 96, 128 and 192 rows a tile cease to make one round over 256 CUs, many rows of narrow weights
    among it: the bits of the kernel that stages tiles through registers."""
    from sonicboom_amd import ops
    k = 448
    packed = ops.pack_weight(randn(2 * inner, k, seed=k, scale=0.05).to(DEV, BF16), True)
    for t in sorted({n + d for n in rows for d in (0, 1)}):
        x = randn(t, k, seed=t).to(DEV, BF16)
        got = ops.gemm_bf16(x, packed, None, None, F32, gated="silu", packed_shape=(2 * inner, k))
        with ops.gemm_tile_shape(0, "registers"):
            want = ops.gemm_bf16(x, packed, None, None, F32, gated="silu", packed_shape=(2 * inner, k))
        assert torch.equal(got, want), t


@pytest.mark.parametrize("count", [1, 2, 15, 16, 17, 32, 33, 64, 65, 255, 256])
def test_top_p_that_ends_on_either_side_of_a_run(count):
    """Shares that the first, the last and the candidates around every sixteenth reach exactly, just not, and just."""
    from plain import sampling_plain as SP
    from sonicboom_amd import ops
    z = (-0.02 * np.arange(count)).astype(np.float32)
    ids = np.random.default_rng(count).permutation(5000)[:count].astype(np.int32)
    e = np.exp(z.astype(np.float64) - float(z[0]))
    shares = np.cumsum(e) / np.cumsum(e)[-1]
    seed, positions = 99, [3, 4000, 77]
    on_gpu = [torch.from_numpy(np.repeat(a[None], 3, 0).copy()).to(DEV) for a in (ids, z)]
    for c in sorted({i for i in (0, 14, 15, 16, 17, 31, 32, 63, 64, count - 2, count - 1) if 0 <= i < count}):
        for share in (shares[c], np.nextafter(shares[c], 0.0), np.nextafter(shares[c], 1.0)):
            top_p = float(np.float32(share))
            if not 0.0 < top_p < 1.0:
                continue
            kept = SP.filter_candidates(list(zip(ids.tolist(), z.tolist())), 0, top_p, 0.0)
            got = ops.draw(*on_gpu, positions, 0, None, top_p, seed).tolist()
            assert got == [SP.draw(kept, seed, p) for p in positions], (c, top_p)


@pytest.mark.parametrize("vocab", [900, 16384, 40003])
def test_candidates_of_rows_alike_spread_and_masked(vocab):
    """Logits of a few values, over many orders, and all but a few of them masked: waves that count by votes and waves that stop."""
    from plain import sampling_plain as SP
    from sonicboom_amd import ops
    g = np.random.default_rng(vocab)
    rows = np.stack([np.zeros(vocab), g.integers(0, 3, vocab) * 0.5, g.standard_normal(vocab) * 10.0 ** g.integers(-6, 5, vocab),
                     np.where(g.random(vocab) < 0.01, g.standard_normal(vocab), -1.0e30), g.standard_normal(vocab)]).astype(np.float32)
    ids, z = ops.top_candidates(torch.from_numpy(rows).to(DEV), 0.7, 256)
    for r, row in enumerate(rows):
        want = SP.select_candidates(row, 0.7)
        assert [c[0] for c in want] == ids[r].tolist() and [np.float32(c[1]) for c in want] == z[r].tolist(), r


def xielu(z, p, q):
    z = z.double().numpy()
    rise, bend = np.log1p(np.exp(p)), 0.5 + np.log1p(np.exp(q))
    return np.where(z > 0, rise * z * z + z / 2, bend * (np.expm1(np.minimum(z, 0.0)) - np.minimum(z, 0.0)) + z / 2)


@pytest.mark.parametrize("n", [3, 4096, (1 << 23) + 5])
def test_xielu_against_64_bits(n):
    """One group of four a thread and several, a tail; numbers around the two borders of its exponential."""
    from sonicboom_amd import ops
    z = randn(n, seed=n, scale=3.0)
    z[:3] = torch.tensor([-1.0, -1e-3, -0.99999994])
    z[n // 2:] *= 0.02
    p = torch.tensor([0.4, -0.3])
    got = ops.activate(z.to(DEV), F32, "xielu", p.to(DEV)).cpu().numpy().astype(np.float64)
    want = xielu(z, 0.4, -0.3)
    # some eight roundings of terms that the result and z / 2 bound
    assert (np.abs(got - want) <= 8 * 2.0 ** -23 * (np.abs(want) + np.abs(z.numpy()))).all()


@pytest.mark.parametrize("n", [12, (1 << 23) + 4])
def test_xielu_of_numbers_that_are_not_finite(n):
    """NaN and minus infinity give a NaN (infinity less infinity), infinity stays, zeros of either sign give zero, and the smallest and the
    largest numbers below zero what 64 bits give."""
    from sonicboom_amd import ops
    z = torch.zeros(n)
    z[:9] = torch.tensor([float("nan"), float("inf"), float("-inf"), -0.0, 0.0, -1.0e-38, -1.0e-20, -200.0, -1.0e30])
    got = ops.activate(z.to(DEV), F32, "xielu", torch.tensor([0.4, -0.3], device=DEV)).cpu()
    assert torch.isnan(got[0]) and got[1] == float("inf") and torch.isnan(got[2]) and (got[3:5] == 0).all() and (got[9:] == 0).all()
    want = torch.from_numpy(xielu(z[5:9], 0.4, -0.3))
    assert ((got[5:9].double() - want).abs() <= 8 * 2.0 ** -23 * (want.abs() + z[5:9].abs())).all()


@pytest.mark.parametrize("t, n, k", [(4001, 4096, 128), (4096, 4094, 192), (4001, 8192, 320)])
def test_xielu_on_a_products_way_out(t, n, k):
    """The bits of the product followed by the pass."""
    from sonicboom_amd import ops
    x, w, p = randn(t, k, seed=1).to(BF16).to(DEV), randn(n, k, seed=2, scale=0.1).to(BF16).to(DEV), torch.tensor([0.4, -0.3], device=DEV)
    packed = ops.pack_weight(w)
    with ops.gemm_tile_shape(2, "direct"):
        z = ops.gemm_bf16(x, packed, None, None, F32, packed_shape=(n, k))
    for dtype in (BF16, F32):
        got = ops.gemm_bf16_activated(x, packed, None, dtype, "xielu", (n, k), params=p)
        assert got is not None and torch.equal(got, ops.activate(z, dtype, "xielu", p))
    assert ops.gemm_bf16_activated(x, packed, torch.zeros(n, device=DEV), BF16, "xielu", (n, k), params=p) is None
    assert ops.gemm_bf16_activated(x[:100], packed, None, BF16, "xielu", (n, k), params=p) is None

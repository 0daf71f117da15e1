"""Latent attention of prompts over built keys and values: the kernels against 64-bit arithmetic, and the plan that the
host lays out for them."""
import numpy as np
import pytest
import torch

BF16 = torch.bfloat16
DEV = "cuda:0"
DIM, ROT, VDIM = 128, 64, 128


def rand(*shape, seed=0, scale=1.0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale


def reference(q_plain, q_rot, rows, uk, uv, cached, window, scale, gate):
    """(want, bound) in 64 bits for one sequence: keys and values rounded to bfloat16 as the product leaves them.
    bound: weights rounded to bfloat16 (2^-9 of each) and the result (2^-9), twice that for products one rounding apart."""
    n, heads = q_plain.shape[:2]
    keys = (rows[:, :-ROT].float() @ uk.float().T).to(BF16).double().reshape(len(rows), heads, DIM)
    values = (rows[:, :-ROT].float() @ uv.float().T).to(BF16).double().reshape(len(rows), heads, VDIM)
    s = (torch.einsum("tad,sad->ats", q_plain.double(), keys) + torch.einsum("tar,sr->ats", q_rot.double(), rows[:, -ROT:].double())) * scale
    t, j = torch.arange(cached, cached + n)[:, None], torch.arange(len(rows))[None, :]
    seen = (j <= t) & ((t - j < window) if window else torch.ones_like(j, dtype=torch.bool))
    p = torch.softmax(s.masked_fill(~seen, float("-inf")), dim=-1)
    g = 1.0 if gate is None else torch.sigmoid(gate.double()).reshape(n, heads, -1)
    want = torch.einsum("ats,sav->tav", p, values) * g
    return want, 2.0 ** -8 * torch.einsum("ats,sav->tav", p, values.abs()) * g + 2.0 ** -8 * want.abs()


@pytest.mark.gpu
@pytest.mark.parametrize("heads, rank, gates", [(1, 512, "number"), (5, 40, "off16"), (16, 256, "head"), (3, 512, None)])
@pytest.mark.parametrize("window", [0, 64, 129])
def test_built_attention_equals_64_bits(heads, rank, gates, window):
    """Runs of one row, of whole tiles, one more and one less; rows that start and end on a page's first and last slot, an odd and an
    even count of pages; a page that is not there; slots that no row sees hold anything, a NaN among it."""
    from sonicboom_amd import ops
    from sonicboom_amd.ops import kernels, library
    from sonicboom_amd.parts.linear import Linear
    assert library.core().sb_built_tile_rows() == kernels.BUILT_ROW_TILE          # the plan lays out what a block takes
    latent, scale = rank + ROT, (DIM + ROT) ** -0.5
    seqs = [(0, 1), (0, 64), (63, 17), (190, 66), (511, 129), (0, 128), (300, 127)]           # (cached keys, rows)
    n_pages = [(k + n + 63) // 64 for k, n in seqs]
    table = torch.full((len(seqs), max(n_pages) + 1), -1, dtype=torch.int32)
    order, at = torch.randperm(sum(n_pages), generator=torch.Generator().manual_seed(2)), 0
    for i, n in enumerate(n_pages):
        table[i, :n] = order[at:at + n].int()
        at += n
    cache = rand(sum(n_pages), 64, latent, seed=3).to(BF16)
    total = sum(n for _, n in seqs)
    q_plain, q_latent = rand(total, heads, DIM, seed=4).to(BF16), rand(total, heads, latent, seed=5).to(BF16)
    uk, uv = rand(heads * DIM, rank, seed=6, scale=rank ** -0.5).to(BF16), rand(heads * VDIM, rank, seed=7, scale=rank ** -0.5).to(BF16)
    wide, per_head = rand(total, heads * VDIM + 16, seed=8), gates == "head"
    gate = {"number": wide[:, 8:8 + heads * VDIM], "off16": wide[:, 3:3 + heads * VDIM], "head": wide[:, :heads], None: None}[gates]
    want, bound, row0 = [], [], 0
    for i, (k, n) in enumerate(seqs):
        rows = cache[table[i, :n_pages[i]].long()].reshape(-1, latent)[:k + n]
        g = None if gate is None else gate[row0:row0 + n]
        w, b = reference(q_plain[row0:row0 + n], q_latent[row0:row0 + n, :, rank:], rows, uk, uv, k, window, scale, g)
        want.append(w)
        bound.append(b)
        row0 += n
    held = cache.clone()
    for i, (k, n) in enumerate(seqs):                    # what nobody sees
        flat = held[table[i, n_pages[i] - 1].long()]
        flat[(k + n - 1) % 64 + 1:] = float("nan")
        if window and k >= window:
            for j in range(k - window + 1):
                held[table[i, j // 64].long(), j % 64] = float("inf")
            if (k - window + 1) // 64 > 0:
                table[i, 0] = -1                          # a page that has gone
    tiles, pages = ops.latent_built_plan([n for _, n in seqs], [k for k, _ in seqs], window)
    build = Linear(torch.cat([uk, uv]).to(DEV), None, True)
    dev = [t.to(DEV) for t in (held, table, torch.from_numpy(tiles), torch.from_numpy(pages))]
    g = None if gate is None else wide.to(DEV)[:, {"number": 8, "off16": 3, "head": 0}[gates]:][:, :gate.shape[1]]
    got = ops.latent_built_attention(q_plain.to(DEV), q_latent.to(DEV), lambda c: build(c, BF16), dev[0], dev[1], dev[2], dev[3], rank, VDIM,
                                     scale, window, g, per_head).double().cpu()
    assert bool(((got - torch.cat(want)).abs() <= torch.cat(bound) + 1e-6).all())


def finite_moves(s, at, window):
    """How often the kernel's running maximum (in powers of two; a half of the waves takes every second page of a tile of 128 rows) moves from
    a finite number, for scores s [rows, keys] of rows at positions ``at``."""
    moves = 0
    for t0 in range(0, len(at), 128):
        lo = max(int(at[t0]) - window + 1, 0) if window else 0
        last = int(at[min(t0 + 127, len(at) - 1)]) // 64
        for half in range(2):
            m = torch.full((min(128, len(at) - t0),), float("-inf"), dtype=torch.float64)
            for page in range(lo // 64 + half, last + 1, 2):
                mx = s[t0:t0 + 128, 64 * page:64 * page + 64].amax(-1) * 1.4426950408889634
                move = mx > m + 8
                moves += int((move & torch.isfinite(m)).sum())
                m = torch.where(move, mx, m)
    return moves


@pytest.mark.gpu
@pytest.mark.parametrize("window", [0, 200])
def test_built_attention_of_peaked_scores(window):
    """Scores that climb by twelve powers of two a page for some rows, fall for others and stay for others still; and, a head on, keys
    that stand out in every second page alone: maxima that move from a finite number, in some lanes of a wave and not in others, and
    halves of a block whose maxima are far apart."""
    from sonicboom_amd import ops
    from sonicboom_amd.parts.linear import Linear
    heads, rank, cached, n, scale = 3, 64, 190, 330, 0.07
    keys = cached + n
    pages_n = (keys + 63) // 64
    cache = rand(pages_n * 64, rank + ROT, seed=3, scale=0.5)
    page, step = torch.arange(pages_n * 64) // 64, 12 * np.log(2) / scale
    cache[:, rank] = step / 16 * page.float()
    cache[:, rank + 1], cache[:, rank + 2] = (page % 2).float() * step / 4, (page % 2 == 0).float() * step / 4
    cache = cache.to(BF16).reshape(pages_n, 64, rank + ROT)
    q_plain, q_latent = rand(n, heads, DIM, seed=4).to(BF16), rand(n, heads, rank + ROT, seed=5)
    row = torch.arange(n)
    q_latent[:, :, rank:rank + 3] = 0.0
    q_latent[:, 0, rank] = torch.tensor([16.0, -16.0, 0.0])[row % 3]
    q_latent[:, 1, rank + 1], q_latent[:, 1, rank + 2] = (row % 2) * 16.0, (row % 4 == 0) * 16.0
    q_latent[:, 2, rank], q_latent[:, 2, rank + 1] = (row % 5 == 0) * 8.0, (row % 3 == 0) * -16.0
    q_latent = q_latent.to(BF16)
    uk, uv = rand(heads * DIM, rank, seed=6, scale=rank ** -0.5).to(BF16), rand(heads * VDIM, rank, seed=7, scale=rank ** -0.5).to(BF16)
    rows = cache.reshape(-1, rank + ROT)[:keys]
    want, bound = reference(q_plain, q_latent[:, :, rank:], rows, uk, uv, cached, window, scale, None)
    # a score is 192 products added in float32, each rounding half a unit of what their absolute values add up to
    k = (rows[:, :rank].float() @ uk.float().T).to(BF16).double().reshape(keys, heads, DIM)
    terms = torch.einsum("tad,sad->ats", q_plain.double().abs(), k.abs()) + torch.einsum("tar,sr->ats", q_latent[:, :, rank:].double().abs(), rows[:, rank:].double().abs())
    bound = bound * (1.0 + 2.0 ** 8 * 2 * 192 * 2.0 ** -24 * float(terms.max()) * scale)
    s = (torch.einsum("tad,sad->ats", q_plain.double(), k) + torch.einsum("tar,sr->ats", q_latent[:, :, rank:].double(), rows[:, rank:].double())) * scale
    at, j = torch.arange(cached, keys), torch.arange(keys)
    seen = (j[None] <= at[:, None]) & ((at[:, None] - j[None] < window) if window else torch.ones(n, keys, dtype=torch.bool))
    moves = [finite_moves(s[a].masked_fill(~seen, float("-inf")), at, window) for a in range(heads)]
    assert moves[0] > 30 and moves[2] > 30, moves            # (head 1: a half of the waves has the pages that stand out)
    tiles, pages = (torch.from_numpy(t).to(DEV) for t in ops.latent_built_plan([n], [cached], window))
    build = Linear(torch.cat([uk, uv]).to(DEV), None, True)
    got = ops.latent_built_attention(q_plain.to(DEV), q_latent.to(DEV), lambda c: build(c, BF16), cache.to(DEV), torch.arange(pages_n, device=DEV).int()[None],
                                     tiles, pages, rank, VDIM, scale, window).double().cpu()
    assert bool(((got - want).abs() <= bound + 1e-6).all())


@pytest.mark.gpu
@pytest.mark.parametrize("number", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("window", [0, 64, 130])
def test_a_number_that_is_not_finite_reaches_the_rows_that_see_it(window, number):
    """A latent with such a number among the keys of a prompt's own tiles: the rows that do not see it keep their bits, the others
    have nothing else."""
    from sonicboom_amd import ops
    from sonicboom_amd.parts.linear import Linear
    heads, rank, cached, n = 2, 64, 70, 300
    table = torch.randperm(6, generator=torch.Generator().manual_seed(1)).int()[None]
    cache = rand(6, 64, rank + ROT, seed=3).to(BF16)
    q_plain, q_latent = rand(n, heads, DIM, seed=4).to(BF16).to(DEV), rand(n, heads, rank + ROT, seed=5).to(BF16).to(DEV)
    build = Linear(rand(2 * heads * DIM, rank, seed=6, scale=rank ** -0.5).to(BF16).to(DEV), None, True)
    tiles, pages = (torch.from_numpy(t).to(DEV) for t in ops.latent_built_plan([n], [cached], window))
    run = lambda c: ops.latent_built_attention(q_plain, q_latent, lambda x: build(x, BF16), c.to(DEV), table.to(DEV), tiles, pages, rank, VDIM,
                                               0.07, window)
    clean = run(cache)
    assert torch.isfinite(clean.float()).all()
    at = torch.arange(cached, cached + n)
    for key in (3, 69, 70, 100, 127, 128, 197, 198, 250, 319, 369):
        for number_of_row in (5, rank + 7):                       # of c, of the rotated part
            if number_of_row >= rank and number != number or number_of_row < rank:
                held = cache.clone()
                held[table[0, key // 64].long(), key % 64, number_of_row] = number
                got = run(held)
                sees = ((at >= key) & ((at - key < window) if window else (at >= 0))).to(DEV)
                assert torch.equal(got[~sees], clean[~sees]), (key, number_of_row)
                assert not torch.isfinite(got[sees].float()).any(), (key, number_of_row)


@pytest.mark.parametrize("window", [0, 64, 200])
def test_plan_covers_every_row_and_every_key_it_sees(window):
    from sonicboom_amd.ops import kernels as K
    n_new, before = [1, 128, 129, 300, 64], [0, 5, 63, 1000, 640]
    tiles, pages = K.latent_built_plan(n_new, before, window)
    rows = sorted((int(r) + i) for r, n, *_ in tiles for i in range(n))
    assert rows == list(range(sum(n_new))) and tiles[:, 1].max() <= K.BUILT_ROW_TILE
    first_row = np.concatenate([[0], np.cumsum(n_new)])
    for r, n, seq, key0, pos, *_ in tiles:
        assert pos == before[seq] + r - first_row[seq]
        lo = max(pos - window + 1, 0) if window else 0
        for j in range(lo, pos + n):                      # the built row of key j is that key's, and not left out
            s, pg, a, b = pages[(key0 + j) // 64]
            assert (s, pg) == (seq, j // 64) and a <= j % 64 < b
    # far more rows than keys: built; single rows on many keys: not; nor what would take too much memory
    sizes = (16, 128, 64, 128, 512)
    assert K.latent_built_pays([2000], [0], 0, *sizes) and not K.latent_built_pays([1, 4], [9000, 9000], 0, *sizes)
    assert not K.latent_built_pays([3000] * 200, [0] * 200, 0, *sizes)

"""The bf16-piece prompt attention (attn_bf16x3.hip) behind ikv_attn_prefill_f32:
every configuration it has, at rows, keys and head sizes off its tiles, against
a 64-bit softmax; paged caches bit for bit; values the pieces do not carry."""
import math

import pytest
import torch

import ikv
from ikv import synth

pytestmark = pytest.mark.gpu


def dev_t(seed, shape, dev, std=1.0):
    return torch.from_numpy(synth.normal(seed, shape, std)).to(dev)


def attn64(q, k, v, past):
    n, H, D = q.shape
    rows, KV, _ = k.shape
    q, k, v = q.double(), k.double(), v.double()
    out = torch.empty_like(q)
    hidden = (torch.arange(rows, device=q.device)[None] >
              past + torch.arange(n, device=q.device)[:, None])
    for h in range(H):
        s = (q[:, h] @ k[:, h * KV // H].t().contiguous()) / math.sqrt(D)
        out[:, h] = torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ v[:, h * KV // H].contiguous()
    return out


# n_q, n_past, query heads, KV heads, head_dim
SHAPES = [
    (300, 0, 16, 8, 128),      # 64-row blocks, two key groups
    (2048, 1, 16, 2, 128),     # a group of 8, one key in the cache
    (513, 4095, 32, 8, 128),   # 128-row blocks, one key group; sums set aside
    (2049, 0, 32, 8, 128),     # ... ragged in rows and keys
    (259, 40, 64, 64, 128),    # a group of 1
    (97, 0, 12, 4, 64),        # 32-row blocks, four key groups, one row of keys past a tile
    (1000, 17, 12, 4, 64),
    (3001, 0, 12, 4, 64),      # two workgroups on a CU
    (130, 70, 6, 1, 96), (200, 0, 10, 5, 80), (500, 0, 12, 4, 32), (333, 9, 4, 2, 4),
    (100, 0, 3, 3, 12), (1, 99, 10, 5, 80), (200, 0, 12, 4, 128),
    # many blocks of few keys, in either form; the last before and the first past the switch
    (140, 0, 64, 64, 64), (200, 0, 128, 128, 32), (150, 0, 40, 40, 128), (95, 0, 128, 128, 64), (96, 0, 128, 128, 64),
    (288, 0, 96, 12, 128), (289, 0, 96, 12, 128),
]


@pytest.mark.parametrize("n,past,H,KV,D", SHAPES)
def test_against_64_bits(dev, n, past, H, KV, D):
    q, k, v = (dev_t(50 + i + n, s, dev) for i, s in
               enumerate(((n, H, D), (n + past, KV, D), (n + past, KV, D))))
    got, ref = ikv.attn_prefill(q, k, v, past), attn64(q, k, v, past)
    assert bool(((got.double() - ref).abs() <= 1e-5 + 1e-4 * ref.abs()).all())
    # F32 sums of P V over n keys: 2^-24 sqrt(keys) of the result, twice for
    # the scores' own rounding
    assert float((got.double() - ref).norm() / ref.norm()) <= 2 ** -23 * (8 + math.sqrt(n + past))
    assert torch.equal(got, ikv.attn_prefill(q, k, v, past))
    # the rows of a prompt do not depend on what follows them in the batch
    wide = torch.cat((k, k.flip(0))), torch.cat((v, v.flip(0)))
    assert torch.equal(got, ikv.attn_prefill(q, *wide, past, n_kv=n + past))


@pytest.mark.parametrize("n,past,H,KV,D,block", [(300, 700, 16, 8, 128, 64), (700, 900, 32, 8, 128, 256),
                                                 (150, 333, 12, 4, 64, 64), (2100, 0, 12, 4, 64, 128),
                                                 # more than 64 blocks
                                                 (300, 8200, 16, 8, 128, 64), (777, 3500, 32, 8, 128, 64),
                                                 (150, 4300, 12, 4, 64, 64), (2100, 2200, 12, 4, 64, 64)])
def test_paged_equals_contiguous(dev, n, past, H, KV, D, block):
    rows = n + past
    q, k, v = (dev_t(70 + i + n, s, dev) for i, s in enumerate(((n, H, D), (rows, KV, D), (rows, KV, D))))
    blocks = -(-rows // block)
    g = torch.Generator(device=dev)
    g.manual_seed(n)
    table = torch.randperm(blocks + 3, generator=g, device=dev)[:blocks].to(torch.int32)
    at = (table.long()[:, None] * block + torch.arange(block, device=dev)).reshape(-1)[:rows]
    pools = []
    for t in (k, v):
        pools.append(torch.full(((blocks + 3) * block, KV, D), float("nan"), device=dev))
        pools[-1][at] = t
    assert torch.equal(ikv.attn_prefill(q, k, v, past),
                       ikv.attn_prefill_paged(q, *pools, table, block, past))


@pytest.mark.parametrize("n,H,KV,D", [(400, 16, 8, 128), (2300, 32, 8, 128), (400, 12, 4, 64), (2500, 12, 4, 64)])
def test_values_the_pieces_cannot_carry(dev, n, H, KV, D):
    q, k, v = (dev_t(90 + i, s, dev) for i, s in enumerate(((n, H, D), (n, KV, D), (n, KV, D))))
    q[:, :, 0] = q[:, :, 0].abs() + 0.5
    base = attn64(q, k, v, 0)
    # an infinite value reaches the rows that see its key, in its own dim only
    v2 = v.clone()
    v2[192, 1, 3] = float("inf")
    got = ikv.attn_prefill(q, k, v2, 0)
    G = H // KV
    hit = torch.zeros_like(base, dtype=torch.bool)
    hit[192:, G:2 * G, 3] = True
    assert bool((got[hit] == float("inf")).all())
    assert bool(((got.double() - base).abs() <= 1e-5 + 1e-4 * base.abs())[~hit].all())
    # a key of -inf (or of a magnitude bf16 rounds to it) in a dim where every
    # query is positive scores -inf and drops out
    for big in (float("-inf"), -3.4e38):
        k2 = k.clone()
        k2[100, 0] = 0
        k2[100, 0, 0] = big
        q2 = q.clone()
        if math.isfinite(big):
            q2[:, :, 0] = q2[:, :, 0] * 4  # the score overflows
        got = ikv.attn_prefill(q2, k2, v, 0)
        k3 = k2.clone()
        k3[100, 0, 0] = -1e30
        want = attn64(q2, k3, v, 0)
        assert bool(((got.double() - want).abs() <= 1e-5 + 1e-4 * want.abs()).all()), big
    # a NaN key makes every row that sees it NaN and no other
    k2 = k.clone()
    k2[300, KV - 1, 5] = float("nan")
    got = ikv.attn_prefill(q, k2, v, 0)
    assert bool(got[300:, H - G:].isnan().all())
    assert not bool(got[:300].isnan().any()) and not bool(got[:, :H - G].isnan().any())
    # values near the bottom of F32's range
    for ex in (-100, -120):
        got = ikv.attn_prefill(q, k, v * 2.0 ** ex, 0)
        assert float((got.double() * 2.0 ** -ex - base).norm() / base.norm()) < 1e-5


@pytest.mark.parametrize("n,past,H,KV,D", [
    (100, 0, 12, 4, 64), (1000, 17, 12, 4, 64), (2501, 0, 12, 4, 64), (150, 3, 10, 5, 80),
    (300, 5, 16, 8, 128), (2050, 0, 32, 8, 128), (1, 99, 10, 5, 80),
    # prompts of the F32 MFMA kernel, in one, two and four wave groups
    (1, 0, 16, 8, 128), (37, 0, 16, 8, 128), (77, 1000, 16, 8, 128), (200, 3, 32, 8, 128), (600, 0, 8, 1, 128)])
def test_rows_behind_the_prompt_are_not_read(dev, n, past, H, KV, D):
    # a longer cache whose later rows hold no numbers: in the last tile of
    # keys, and past it
    q, k, v = (dev_t(110 + i + n, s, dev) for i, s in
               enumerate(((n, H, D), (n + past, KV, D), (n + past, KV, D))))
    want = ikv.attn_prefill(q, k, v, past)
    block = 64
    rows = -(-(n + past + 150) // block) * block
    for what in ("nan", "inf"):
        caches = []
        for t in (k, v):
            caches.append(torch.full((rows, KV, D), float(what), device=dev))
            caches[-1][:n + past] = t
        assert torch.equal(ikv.attn_prefill(q, *caches, past, n_kv=rows), want)
        table = torch.arange(rows // block, dtype=torch.int32, device=dev)
        assert torch.equal(ikv.attn_prefill_paged(q, *caches, table, block, past, n_kv=rows), want)


@pytest.mark.parametrize("n,H,KV,D", [(400, 16, 8, 128), (2300, 32, 8, 128), (400, 12, 4, 64), (2500, 12, 4, 64)])
@pytest.mark.parametrize("key", [0, 203, 319])
def test_a_value_that_is_no_number_reaches_no_earlier_row(dev, n, H, KV, D, key):
    q, k, v = (dev_t(120 + i, s, dev) for i, s in enumerate(((n, H, D), (n, KV, D), (n, KV, D))))
    base = attn64(q, k, v, 0)
    G = H // KV
    for bad in (float("inf"), float("nan")):
        v2 = v.clone()
        v2[key, 1, 3] = bad
        got = ikv.attn_prefill(q, k, v2, 0)
        hit = torch.zeros_like(base, dtype=torch.bool)
        hit[key:, G:2 * G, 3] = True
        assert bool((got[hit].isnan() if bad != bad else got[hit] == bad).all())
        assert bool(((got.double() - base).abs() <= 1e-5 + 1e-4 * base.abs())[~hit].all())
        # the wave that starts over sums in another order, not with fewer bits
        assert float((got.double() - base)[~hit].norm() / base[~hit].norm()) <= 2 ** -23 * (8 + math.sqrt(n))


@pytest.mark.parametrize("n,past,H,KV,D", [(400, 0, 16, 8, 128), (2300, 0, 32, 8, 128), (400, 7, 12, 4, 64),
                                           (2500, 0, 12, 4, 64)])
def test_small_floats_keep_their_bits_beside_ordinary_ones(dev, n, past, H, KV, D):
    # a float below 2^-109 has bits that no bf16 piece holds: dims, keys and
    # whole values of them, queries of them against large keys and keys of them
    # against large queries. Dim by dim and head by head as far from 64 bits as
    # F32 sums are
    q, k, v = (dev_t(130 + i, s, dev) for i, s in
               enumerate(((n, H, D), (n + past, KV, D), (n + past, KV, D))))
    bar = 2 ** -23 * (8 + math.sqrt(n + past))

    def check(q, k, v, what, bar=bar):
        got, ref = ikv.attn_prefill(q, k, v, past).double(), attn64(q, k, v, past)
        floor = n * 2.0 ** -149  # of denormal results
        assert bool(((got - ref).norm(dim=0) <= bar * ref.norm(dim=0) + floor).all()), what

    for ex in (-109, -115, -122, -128):
        v2 = v.clone()
        v2[:, :, 5] *= 2.0 ** ex
        check(q, k, v2, ("dim", ex))
        check(q, k, v * 2.0 ** ex, ("values", ex))
        check(q * 2.0 ** ex, k * 2.0 ** min(-ex, 120), v, ("queries", ex))
        k2, q2 = k.clone(), q.clone()
        k2[:, :, 7] *= 2.0 ** ex
        q2[:, :, 7] *= 2.0 ** min(-ex, 120)
        check(q2, k2, v, ("keys", ex))


@pytest.mark.parametrize("n,H,KV,D", [(400, 16, 8, 128), (2300, 32, 8, 128), (400, 12, 4, 64), (2500, 12, 4, 64)])
@pytest.mark.parametrize("nats", [70, 80, 86])
def test_small_probabilities_keep_their_bits(dev, n, H, KV, D, nats):
    # key 0 takes nearly all the weight and its value is zero: a row is the sum
    # of the others' weights near e^-nats (2^-101, 2^-115, 2^-124)
    q, k, v = (dev_t(140 + i, s, dev) for i, s in enumerate(((n, H, D), (n, KV, D), (n, KV, D))))
    q *= 0.1
    q[:, :, 0] = math.sqrt(D)
    k[:, :, 0] = -float(nats)
    k[0] = 0
    v = v.abs()
    v[0] = 0
    got, ref = ikv.attn_prefill(q, k, v, 0).double(), attn64(q, k, v, 0)
    # a score of this size is rounded to 2^-24 of it at each of its sum's D / 16
    # matrix steps (the first dim puts it there), where the two parts of the sum
    # meet, at its scale and at its distance from the largest; pieces that
    # drop bits below 2^-133 are off by 2^-9 at 86
    bar = (D / 16 + 3) * nats * 2 ** -24 + 2 ** -23 * (8 + math.sqrt(n))
    assert bool(((got - ref).norm(dim=2) <= bar * ref.norm(dim=2)).all())

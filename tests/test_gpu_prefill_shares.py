"""Prompt chunks whose (chunk, KV head) pairs are no multiple of the XCDs: each pair's query tiles are dealt to several of
them in turn. Every tile of every pair has to be computed once, whatever the pairs' count and the tiles' remainder: the
rows at the tiles' edges against float64 attention over the stored values, all rows against the chunk launched alone."""
import pytest
import torch

from tests.support import Cache, rand_q

pytestmark = pytest.mark.gpu
dev = "cuda"
# 16-bit probabilities and results: 2^-8 of the largest weight and of the result, four times that
ATOL, RTOL = 8e-3, 2e-2


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("hkv,chunks", [(1, 1), (2, 1), (3, 1), (4, 1), (3, 2), (1, 4), (2, 4), (3, 3)])
def test_every_tile_of_every_pair_is_computed(hkv, chunks, d):
    g = 3
    counts = [(1, 43, 300, 129)[i] for i in range(chunks)]      # 3 to 900 rows of a pair: under a tile, one row over, ragged
    prefix = [(20, 0, 65, 7)[i] for i in range(chunks)]
    cache = Cache("bf16", hkv, d, d, 16, [p + n for p, n in zip(prefix, counts)], seed=hkv)
    q = rand_q(sum(counts), g * hkv, d, 4).bfloat16()
    starts = [sum(counts[:i]) for i in range(chunks)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    i64 = lambda x: torch.tensor(x, dtype=torch.int64, device=dev)
    pk = cache.pk
    out = pk.prefill_rows(q, cache.k, cache.v, "bf16", cache.tables, i32(list(range(chunks))), i32(starts), i32(counts), i64(prefix),
                          max(counts), 16)
    for s, (start, n, first) in enumerate(zip(starts, counts, prefix)):
        alone = pk.prefill_rows(q[start:start + n], cache.k, cache.v, "bf16", cache.tables, i32([s]), i32([0]), i32([n]), i64([first]), n, 16)
        assert torch.equal(alone, out[start:start + n]), s
        for t in sorted({0, 42, 43, n // 2, n - 1} & set(range(n))):
            want, _ = cache.want(q[start + t:start + t + 1], s, first + t, 1)
            torch.testing.assert_close(out[start + t:start + t + 1].double().cpu(), want, atol=ATOL, rtol=RTOL, msg=f"{s} {t}")


def _prefill(cache, q, counts, prefix, fresh=None, **kw):
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    starts = [sum(counts[:i]) for i in range(len(counts))]
    return cache.pk.prefill_rows(q, cache.k, cache.v, cache.kind, cache.tables, i32(list(range(len(counts)))), i32(starts), i32(counts),
                                 torch.tensor(prefix, dtype=torch.int64, device=dev), max(counts), 16, key_scales=cache.ks,
                                 value_scales=cache.vs, multipliers=cache.multipliers, fresh=fresh, **kw)


@pytest.mark.parametrize("kind", ["bf16", "fp8", "int8"])
@pytest.mark.parametrize("hkv,g,n", [(2, 16, 2101), (1, 32, 2070), (6, 8, 1400)])
def test_eight_wavefronts_on_pairs_dealt_to_several_xcds(kind, hkv, g, n):
    # 128-wide heads with a tile of 256 rows or more for every compute unit: 2 pairs of 132 tiles, 1 of 259, 6 of 44
    first = 37
    cache = Cache(kind, hkv, 128, 128, 16, [first + n], seed=3)
    q = rand_q(n, hkv * g, 128, 5).bfloat16()
    out = _prefill(cache, q, [n], [first])
    for at in range(0, n, 500):      # the same tokens a few at a time: launches of four wavefronts a workgroup
        m = min(500, n - at)
        assert torch.equal(out[at:at + m], _prefill(cache, q[at:at + m], [m], [first + at])), at
    for t in (0, 7, 8, 15, 16, n // 2, n - 1):
        want, _ = cache.want(q[t:t + 1], 0, first + t, 1)
        torch.testing.assert_close(out[t:t + 1].double().cpu(), want, atol=ATOL, rtol=RTOL, msg=str(t))


@pytest.mark.parametrize("kind", ["fp8", "fp8:row", "int8"])
@pytest.mark.parametrize("hkv,chunks", [(1, 1), (2, 1), (1, 3), (4, 3)])
def test_fresh_rows_of_dealt_pairs(kind, hkv, chunks):
    # two launches a call, each with tiles of its own height, over pairs dealt to 8, 4 and 2 XCDs
    counts, prefix = [700, 43, 300][:chunks], [20, 90, 65][:chunks]
    cache = Cache(kind, hkv, 128, 128, 16, [p + n for p, n in zip(prefix, counts)], seed=7)
    q = rand_q(sum(counts), 4 * hkv, 128, 8).bfloat16()
    fk, fv = rand_q(sum(counts), hkv, 128, 9).bfloat16(), rand_q(sum(counts), hkv, 128, 10).bfloat16()
    out = _prefill(cache, q, counts, prefix, fresh=(fk, fv))
    for s, (n, first) in enumerate(zip(counts, prefix)):
        start = sum(counts[:s])
        for t in sorted({0, 31, 32, 42, 127, 128, n // 2, n - 1} & set(range(n))):
            want, _ = cache.want(q[start + t:start + t + 1], s, first + t, 1,
                                 fresh=(fk[start:start + n].cpu(), fv[start:start + n].cpu(), first, first))
            torch.testing.assert_close(out[start + t:start + t + 1].double().cpu(), want, atol=ATOL, rtol=RTOL, msg=f"{s} {t}")


def test_many_pairs_of_short_chunks_beside_a_long_one():
    # 2 KV heads, 33 chunks of 1 to 9 tokens and one of 600: pairs of one live tile in a launch sized for eight times as many
    counts = [1 + i % 9 for i in range(33)]
    counts[11] = 600
    prefix = [5 * i for i in range(33)]
    cache = Cache("bf16", 2, 64, 64, 16, [p + n for p, n in zip(prefix, counts)], seed=11)
    q = rand_q(sum(counts), 4, 64, 12).bfloat16()
    out = _prefill(cache, q, counts, prefix)
    for s, (n, first) in enumerate(zip(counts, prefix)):
        start = sum(counts[:s])
        for t in sorted({0, n // 2, n - 1}):
            want, _ = cache.want(q[start + t:start + t + 1], s, first + t, 1)
            torch.testing.assert_close(out[start + t:start + t + 1].double().cpu(), want, atol=ATOL, rtol=RTOL, msg=f"{s} {t}")

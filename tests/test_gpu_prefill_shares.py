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

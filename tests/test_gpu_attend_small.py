"""Launches of no more units than compute units, a workgroup a unit without a list, which keep two pairs of a wavefront's steps in
flight in LDS, and draft trees, whose ancestors the lanes work out among themselves: against float64 attention and against the
same rows in launches that take the other kernels."""
import pytest
import torch

from tests.support import Cache, rand_q

pytestmark = pytest.mark.gpu
dev = "cuda"
ATOL, RTOL = 8e-3, 2e-2


@pytest.mark.parametrize("kind", ["bf16", "fp16", "fp8", "fp8:row", "int8"])
@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (8, 2, 128), (16, 4, 64), (12, 2, 256), (9, 3, 128)])
@pytest.mark.parametrize("columns", [1, 3, 5, 8])
def test_small_launches_give_the_bits_of_large_ones(kind, hq, hkv, d, columns):
    # contexts around a step (8 positions), a wavefront's first pairs (64, 128), a piece (256 to 1,536) and several
    firsts = [0, 1, 7, 8, 31, 63, 64, 127, 128, 200, 511, 512, 513, 768, 1100, 1536 - columns, 1600]
    cache = Cache(kind, hkv, d, d, 16, [n + columns for n in firsts], seed=hq + d)
    q = rand_q(columns * len(firsts), hq, d, 3)
    starts = [columns * i for i in range(len(firsts))]
    # forty of each row: far more units than compute units
    many = cache.attend(q, list(range(len(firsts))) * 40, starts * 40, firsts * 40, columns)
    for i, first in enumerate(firsts):
        lse = torch.empty(columns, hq, device=dev)
        tables = cache.tables
        cache.tables = tables[:, :-(-(first + columns) // 16)].contiguous()      # (no longer than the row: few units listed)
        alone = cache.attend(q[starts[i]:starts[i] + columns], [i], [0], [first], columns, lse=lse)
        cache.tables = tables
        assert torch.equal(alone, many[starts[i]:starts[i] + columns]), first
        want, want_lse = cache.want(q[starts[i]:starts[i] + columns], i, first, columns)
        torch.testing.assert_close(alone.double().cpu(), want, atol=ATOL, rtol=RTOL)
        torch.testing.assert_close(lse.double().cpu(), want_lse, atol=1e-3, rtol=1e-4)


@pytest.mark.parametrize("kind,hq,hkv,d", [("bf16", 8, 2, 128), ("fp8", 8, 2, 128), ("int8", 4, 1, 128), ("fp8:row", 8, 2, 256)])
@pytest.mark.parametrize("columns", [1, 2, 31, 33, 64])
@pytest.mark.parametrize("links", [torch.int32, torch.int64])
def test_ancestors_of_wide_trees(kind, hq, hkv, d, columns, links):
    # rows of a chain, of a star, of random links, and of links that are none (no earlier column), one of them short
    g = torch.Generator().manual_seed(columns)
    chain = [c - 1 for c in range(columns)]
    star = [-1] + [0] * (columns - 1)
    loose = [int(torch.randint(-1, max(1, c), (), generator=g)) for c in range(columns)]
    wrong = [c if c % 3 == 0 else (columns + 5 if c % 3 == 1 else c - 1) for c in range(columns)]
    if links == torch.int64:
        wrong = [x + (1 << 32) if c % 5 == 4 else x for c, x in enumerate(wrong)]
    trees, firsts = [chain, star, loose, wrong], [40, 0, 700, 17]
    counts = [columns, columns, columns, max(1, columns - 1)]
    cache = Cache(kind, hkv, d, d, 16, [n + columns for n in firsts], seed=7)
    q = rand_q(4 * columns, hq, d, 9)
    out = cache.attend(q, [0, 1, 2, 3], [columns * i for i in range(4)], firsts, columns,
                       counts=torch.tensor(counts, dtype=torch.int32, device=dev),
                       parents=torch.tensor([x for tree in trees for x in tree], dtype=links, device=dev))
    for i, (tree, first, count) in enumerate(zip(trees, firsts, counts)):
        at = slice(columns * i, columns * i + count)
        clean = torch.tensor([x if 0 <= x < c else -1 for c, x in enumerate(tree)][:count], dtype=torch.int32)
        want, _ = cache.want(q[at], i, first, count, parents=clean)
        torch.testing.assert_close(out[at].double().cpu(), want, atol=ATOL, rtol=RTOL)


@pytest.mark.parametrize("kind", ["bf16", "fp16", "fp8", "fp8:row", "int8"])
@pytest.mark.parametrize("lengths", [[9000], [6500, 700], [40, 5000]])
@pytest.mark.parametrize("columns,tree", [(1, False), (3, False), (4, True)])
@pytest.mark.parametrize("d", [128, 64])
def test_one_or_two_rows_of_more_places_than_compute_units(kind, lengths, columns, tree, d):
    # pieces of 64: hundreds of partitions of the heads' wavefronts; the fused launch makes the same bits
    hq, hkv = 32, 8
    cache = Cache(kind, hkv, d, d, 16, lengths, seed=len(lengths))
    n = len(lengths)
    q = rand_q(n * columns, hq, d, 11)
    firsts, starts = [x - columns for x in lengths], [columns * i for i in range(n)]
    given = dict(partitions=200, piece=64)      # (64-wide heads in pairs: two places a partition and tile)
    if tree:
        given["parents"] = torch.tensor([-1, 0, 0, 1] * n, dtype=torch.int32, device=dev)
    lse, again = torch.empty(n * columns, hq, device=dev), torch.empty(n * columns, hq, device=dev)
    out = cache.attend(q, list(range(n)), starts, firsts, columns, lse=lse, **given)
    assert torch.equal(cache.attend(q, list(range(n)), starts, firsts, columns, lse=again, fused=True, **given), out) and torch.equal(lse, again)
    for i, first in enumerate(firsts):
        at = slice(starts[i], starts[i] + columns)
        want, _ = cache.want(q[at], i, first, columns, parents=torch.tensor([-1, 0, 0, 1], dtype=torch.int32) if tree else None)
        torch.testing.assert_close(out[at].double().cpu(), want, atol=ATOL, rtol=RTOL)


@pytest.mark.parametrize("kind", ["bf16", "fp8", "int8"])
@pytest.mark.parametrize("partitions", [30, 50, 120])
@pytest.mark.parametrize("lengths,counts", [([6000, 900], [3, 3]), ([900, 6000], [3, 3]), ([6000, 6000], [3, 2]), ([3300, 6000], [3, 3]), ([4000, 70], [0, 3]),
                                            ([5000, 5000], [3, 0])])
def test_two_uneven_rows_in_partitions_of_one_piece_and_of_several(kind, partitions, lengths, counts):
    # pieces of 64: up to 94 of a row; more places than compute units in one partition a piece and in several pieces a partition
    hq, hkv, d, columns = 32, 8, 128, 3
    cache = Cache(kind, hkv, d, d, 16, lengths, seed=partitions)
    cache.tables = torch.cat([cache.tables, cache.tables[:, :1].expand(2, 500)], 1).contiguous()      # (tables wider than their rows)
    q = rand_q(2 * columns, hq, d, 13)
    firsts, starts = [x - columns for x in lengths], [0, columns]
    given = dict(partitions=partitions, piece=64, counts=torch.tensor(counts, dtype=torch.int32, device=dev))
    results = []
    for fused in (False, True):
        out, lse = torch.zeros(2 * columns, hq, d, device=dev), torch.zeros(2 * columns, hq, device=dev)
        cache.attend(q, [0, 1], starts, firsts, columns, out=out, lse=lse, fused=fused, **given)
        results += [out, lse]
    assert torch.equal(results[0], results[2]) and torch.equal(results[1], results[3])
    for i, (first, count) in enumerate(zip(firsts, counts)):
        at = slice(starts[i], starts[i] + count)
        if count:
            want, _ = cache.want(q[at], i, first, count)
            torch.testing.assert_close(results[0][at].double().cpu(), want, atol=ATOL, rtol=RTOL)

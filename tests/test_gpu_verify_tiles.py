"""Verify windows read three query tiles a workgroup, draft trees whose steps lie before, across and behind the window's
first position, and trees and sliding windows over several rows of fewer columns than the launch: every column against
float64 attention over the stored values and, bit for bit, against its fused launch."""
import pytest
import torch

from tests.support import Cache, rand_q

pytestmark = pytest.mark.gpu
dev = "cuda"
# 16-bit probabilities and results: 2^-8 of the largest weight and of the result, four times that
ATOL, RTOL = 8e-3, 2e-2


@pytest.mark.parametrize("kind", ["bf16", "fp16"])
@pytest.mark.parametrize("hkv,g,columns", [(2, 4, 5), (2, 4, 6), (2, 7, 3), (2, 7, 6), (2, 8, 9), (3, 4, 9), (3, 4, 12), (3, 7, 11)])
def test_windows_of_three_tiles_a_workgroup(kind, hkv, g, columns):
    # 3, 5, 6 and 9 tiles (of 8 rows with two KV heads a wavefront, of 16 with one), the last ones full and not
    cache = Cache(kind, hkv, 128, 128, 16, [1100, 25, 530])
    firsts, counts = [1100 - columns, 25 - columns, 511], [columns, max(1, columns - 2), min(columns, 4)]
    starts = [0, columns, 2 * columns]
    q = rand_q(3 * columns, hkv * g, 128, 31)
    i32 = torch.tensor(counts, dtype=torch.int32, device=dev)
    out = cache.attend(q, [0, 1, 2], starts, firsts, columns, counts=i32)
    fused = cache.attend(q, [0, 1, 2], starts, firsts, columns, counts=i32, fused=True)
    for s, (start, first, n) in enumerate(zip(starts, firsts, counts)):
        assert torch.equal(out[start:start + n], fused[start:start + n]), s
        want, _ = cache.want(q[start:start + n], s, first, n)
        torch.testing.assert_close(out[start:start + n].double().cpu(), want, atol=ATOL, rtol=RTOL, msg=str(s))
        one = cache.attend(q[start + n - 1:start + n], [s], [0], [first + n - 1], 1)
        assert torch.equal(one[0], out[start + n - 1]), s


@pytest.mark.parametrize("kind", ["bf16", "fp8", "fp8:row", "int8"])
@pytest.mark.parametrize("hkv,g,d,columns", [(2, 4, 128, 5), (2, 7, 128, 8), (3, 4, 128, 5), (2, 6, 256, 5), (4, 4, 64, 6)])
@pytest.mark.parametrize("first", [0, 1, 7, 8, 15, 16, 17, 520, 527])
def test_trees_at_every_place_of_the_windows_first_position_in_a_step(kind, hkv, g, d, columns, first):
    cache = Cache(kind, hkv, d, d, 16, [first + columns])
    parents = torch.tensor([-1, 0, 0, 1, 1, 2, 5, 3][:columns], dtype=torch.int32, device=dev)
    q = rand_q(columns, hkv * g, d, 32)
    out = cache.attend(q, [0], [0], [first], columns, parents=parents)
    assert torch.equal(out, cache.attend(q, [0], [0], [first], columns, parents=parents, fused=True))
    chain = cache.attend(q, [0], [0], [first], columns, parents=torch.arange(-1, columns - 1, dtype=torch.int32, device=dev))
    assert torch.equal(chain, cache.attend(q, [0], [0], [first], columns))
    want, _ = cache.want(q.to(torch.bfloat16), 0, first, columns, parents=parents.tolist())
    torch.testing.assert_close(out.double().cpu(), want, atol=ATOL, rtol=RTOL)


@pytest.mark.parametrize("kind", ["bf16", "fp16", "fp8", "fp8:row", "int8"])
@pytest.mark.parametrize("sliding", [0, 33, 300])
@pytest.mark.parametrize("hkv,g,d,columns", [(2, 4, 128, 4), (2, 4, 128, 5), (2, 4, 128, 8), (3, 4, 128, 9), (2, 7, 128, 6), (2, 8, 128, 9), (2, 6, 256, 5), (4, 4, 64, 6)])
def test_trees_and_sliding_windows_over_several_ragged_rows(kind, sliding, hkv, g, d, columns):
    # 1 to 9 tiles, rows of every column and of fewer (dead columns in a tile, tiles without a live row), a tree alone, a
    # sliding window alone and both, split and fused: the same bits, a chain's tree those of the window without one
    counts = [columns, 1, columns - 1, max(1, columns // 2)]
    lengths = [1100, 25, 530, 40 + columns]
    cache = Cache(kind, hkv, d, d, 16, lengths)
    firsts, starts = [n - c for n, c in zip(lengths, counts)], [columns * i for i in range(4)]
    q = rand_q(4 * columns, hkv * g, d, 33)
    i32 = torch.tensor(counts, dtype=torch.int32, device=dev)
    links = [-1, 0, 0, 1, 1, 2, 5, 3, 6][:columns]
    parents = torch.tensor(links * 4, dtype=torch.int32, device=dev)
    chains = torch.arange(-1, columns - 1, dtype=torch.int32, device=dev).repeat(4)
    run = lambda **kw: cache.attend(q, [0, 1, 2, 3], starts, firsts, columns, counts=i32, sliding=sliding, **kw)
    out, fused, chain, plain = run(parents=parents), run(parents=parents, fused=True), run(parents=chains), run()
    for s, (start, first, n) in enumerate(zip(starts, firsts, counts)):
        assert torch.equal(out[start:start + n], fused[start:start + n]), s
        assert torch.equal(chain[start:start + n], plain[start:start + n]), s
        for got, up in ((out, links[:n]), (plain, None)):
            want, _ = cache.want(q[start:start + n], s, first, n, sliding=sliding, parents=up)
            torch.testing.assert_close(got[start:start + n].double().cpu(), want, atol=ATOL, rtol=RTOL, msg=f"{s} {up}")


@pytest.mark.parametrize("columns,g", [(5, 7), (6, 7), (9, 8)])
def test_what_the_caller_says_of_its_columns_changes_no_bit(columns, g):
    # 65 rows of 8 KV heads: enough of them that a launch of five, six or nine tiles takes three a workgroup only where the
    # partial rows say that every row is full; here some are (as packed rows say), some are not (as unpacked ones may be)
    rows = 65
    lengths = [columns + 1 + (7 * r) % 50 for r in range(rows)]
    cache = Cache("bf16", 8, 128, 128, 16, lengths)
    q = rand_q(rows * columns, 8 * g, 128, 34)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    for counts in ([columns] * rows, [columns - r % 3 for r in range(rows)], [1 + r % columns for r in range(rows)]):
        starts, firsts = [columns * r for r in range(rows)], [n - c for n, c in zip(lengths, counts)]
        run = lambda **kw: cache.attend(q, list(range(rows)), starts, firsts, columns, counts=i32(counts), out=torch.zeros_like(q, dtype=torch.bfloat16), **kw)
        plain = run()
        packed = [sum(counts[:r]) for r in range(rows)]
        assert torch.equal(plain, run(offsets=i32(packed), tokens=sum(counts)))
        assert torch.equal(plain, run(offsets=i32(starts), tokens=rows * columns))
        for r in (0, 3, 64):
            want, _ = cache.want(q[starts[r]:starts[r] + counts[r]], r, firsts[r], counts[r])
            torch.testing.assert_close(plain[starts[r]:starts[r] + counts[r]].double().cpu(), want, atol=ATOL, rtol=RTOL, msg=str(r))

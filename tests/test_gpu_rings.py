"""Where the window kernels' pairs of steps, rings, folds and merges, the prompt kernel's loads straight into LDS, the index
selection's short list and shared keys and the latent merge's wide stores can go wrong: pieces whose last pair lacks a step, wavefronts
without a step, units of more pairs than a wavefront holds entries for, three tiles of 8-bit pages, merges of many
wavefronts and of long rows, and edges of lists. Against float64 attention over the stored values, the oracle's picks, or
the fused launch bit for bit."""
import pytest
import torch

from oracle import indexer as oracle_indexer
from tests.support import Cache, kernels, rand_q

pytestmark = pytest.mark.gpu
dev = "cuda"
# 16-bit probabilities and results: 2^-8 of the largest weight and of the result, four times that
ATOL, RTOL = 8e-3, 2e-2

HEADS = [("bf16", 2, 4, 128), ("bf16", 3, 4, 128), ("fp16", 2, 4, 256), ("fp8", 2, 4, 128), ("fp8:row", 2, 6, 256), ("int8", 3, 4, 128), ("int8", 2, 4, 64)]


def close(got, want, **kw):
    torch.testing.assert_close(got.double().cpu(), want, atol=ATOL, rtol=RTOL, **kw)


@pytest.mark.parametrize("kind,hkv,g,d", HEADS)
@pytest.mark.parametrize("parts,piece", [(64, 16), (3, 48), (5, 80), (2, 112), (1, 144), (1, 4608), (2, 2064)])
def test_pieces_that_end_within_a_pair_and_units_of_many_pairs(kind, hkv, g, d, parts, piece):
    # a wavefront's steps of a piece are 1, 2, 3 .. or none; one unit of 4,608 positions is 72 pairs of a wavefront (two heads
    # a wavefront) or 36, past the 32 whose entries it holds, in one piece or in many
    n = 4500
    cache = Cache(kind, hkv, d, d, 16, [n, 37], seed=piece)
    q = rand_q(3, hkv * g, d, 61)
    out = cache.attend(q, [0, 1], [0, 2], [n - 2, 36], 2, counts=torch.tensor([2, 1], dtype=torch.int32, device=dev), partitions=parts, piece=piece)
    fused = cache.attend(q, [0, 1], [0, 2], [n - 2, 36], 2, counts=torch.tensor([2, 1], dtype=torch.int32, device=dev), partitions=parts, piece=piece, fused=True)
    assert torch.equal(out, fused)
    close(out[:2], cache.want(q[:2], 0, n - 2, 2)[0])
    close(out[2:], cache.want(q[2:], 1, 36, 1)[0])


@pytest.mark.parametrize("kind", ["bf16", "fp16", "fp8"])
@pytest.mark.parametrize("scale", [-0.1, 0.0, 2.0])
def test_scales_of_any_sign(kind, scale):
    cache = Cache(kind, 2, 128, 128, 16, [700])
    q = rand_q(2, 8, 128, 62)
    out = cache.attend(q, [0], [0], [698], 2, scale=scale)
    assert torch.equal(out, cache.attend(q, [0], [0], [698], 2, scale=scale, fused=True))
    close(out, cache.want(q, 0, 698, 2, scale=scale)[0])


@pytest.mark.parametrize("kind,hkv,d", [("bf16", 2, 128), ("bf16", 3, 128), ("fp16", 2, 256), ("fp8", 2, 128), ("fp8", 4, 64), ("fp8:row", 2, 128), ("int8", 2, 128)])
@pytest.mark.parametrize("fused", [False, True])
def test_a_scale_that_is_no_number_shows(kind, hkv, d, fused):
    cache = Cache(kind, hkv, d, d, 16, [700])
    q = rand_q(2, 4 * hkv, d, 69)
    assert bool(cache.attend(q, [0], [0], [698], 2, scale=float("nan"), fused=fused).isnan().all())
    if kind == "fp8":      # a head's multiplier: its own query heads, and no others
        want = cache.attend(q, [0], [0], [698], 2, fused=fused)
        per_head = torch.tensor([[0.02] * hkv, [0.03] * hkv])
        per_head[0, 1] = float("nan")
        cache.multipliers = per_head
        out = cache.attend(q, [0], [0], [698], 2, fused=fused)
        assert bool(out[:, 4:8].isnan().all())
        assert torch.equal(out[:, :4], want[:, :4]) and torch.equal(out[:, 8:], want[:, 8:])


@pytest.mark.parametrize("kind", ["fp8", "fp8:row", "int8"])
@pytest.mark.parametrize("tree", [False, True])
@pytest.mark.parametrize("sliding", [0, 33])
@pytest.mark.parametrize("hkv,columns", [(8, 5), (8, 6), (3, 11), (3, 12)])
def test_three_tiles_of_8_bit_pages_in_a_launch_that_fills_the_card(kind, tree, sliding, hkv, columns):
    # 180 rows of 4 pairs of heads (tiles of 8 rows) or of 3 heads (of 16): more than two a compute unit. The rows' columns as
    # the caller leaves them unsaid, and as a verify round says them: counts, and partial rows packed by their offsets
    rows, g = 180, 4
    lengths = [columns + 1 + (11 * r) % 90 for r in range(rows)]
    cache = Cache(kind, hkv, 128, 128, 16, lengths)
    q = rand_q(rows * columns, hkv * g, 128, 63)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    starts, firsts = [columns * r for r in range(rows)], [n - columns for n in lengths]
    links = [-1, 0, 0, 1, 3, 2, 5, 4, 4, 8, 9, 6][:columns] if tree else None
    parents = i32(links * rows) if tree else None
    run = lambda **kw: cache.attend(q, list(range(rows)), starts, firsts, columns, parents=parents, sliding=sliding, **kw)
    out = run()
    assert torch.equal(out, run(fused=True))
    assert torch.equal(out, run(counts=i32([columns] * rows), offsets=i32(starts), tokens=rows * columns))
    for r in (0, 7, 179):
        want, _ = cache.want(q[starts[r]:starts[r] + columns], r, firsts[r], columns, sliding=sliding, parents=links)
        close(out[starts[r]:starts[r] + columns], want, msg=str(r))


@pytest.mark.parametrize("kind,hkv,g,d", [("bf16", 2, 4, 128), ("fp8", 2, 4, 256), ("bf16", 2, 4, 64)])
@pytest.mark.parametrize("n,parts,rows", [(16 * 33, 33, 1), (16 * 128, 128, 1), (16 * 129 - 3, 200, 1), (16 * 257, 300, 1), (16 * 9, 9, 256), (16 * 17 - 5, 17, 300)])
def test_merges_of_long_rows_and_of_many_wavefronts(kind, hkv, g, d, n, parts, rows):
    # a workgroup a triple (more than 32 partitions of few triples; 128 or 256 at a time), and batches of 8 partitions (2,048
    # wavefronts or more): the fused launch's bits, log-sum-exps and sinks too
    cache = Cache(kind, hkv, d, d, 16, [n], seed=parts)
    q = rand_q(rows, hkv * g, d, 64)
    sinks = torch.linspace(-2, 2, hkv * g, device=dev)
    for with_sinks in (None, sinks):
        lse, fused_lse = torch.empty(rows, hkv * g, device=dev), torch.empty(rows, hkv * g, device=dev)
        run = lambda **kw: cache.attend(q, [0] * rows, list(range(rows)), [n - 1] * rows, 1, partitions=parts, piece=16, sinks=with_sinks, **kw)
        out = run(lse=lse)
        assert torch.equal(out, run(lse=fused_lse, fused=True))
        assert torch.equal(lse, fused_lse)
        for r in {0, rows - 1}:
            want, want_lse = cache.want(q[r:r + 1], 0, n - 1, 1)
            if with_sinks is not None:      # a logit more in the sum, with no value
                with_sink = torch.logaddexp(want_lse, sinks.double().cpu())
                want, want_lse = want * torch.exp(want_lse - with_sink)[..., None], with_sink
            close(out[r:r + 1], want, msg=str(r))
            torch.testing.assert_close(lse[r:r + 1].double().cpu(), want_lse, atol=1e-3, rtol=1e-4, msg=str(r))


@pytest.mark.parametrize("hkv,g,d", [(2, 4, 128), (1, 4, 256), (2, 4, 64)])
def test_merges_of_short_rows_in_wide_tables(hkv, g, d):
    # tables with room for 100 partitions: rows of up to 32 go by one wavefront, others by the workgroup, both beside each other
    lengths = [1, 16 * 8, 16 * 8 + 1, 16 * 32, 16 * 32 + 1, 16 * 60 - 5]
    cache = Cache("bf16", hkv, d, d, 16, lengths)
    q = rand_q(2 * len(lengths), hkv * g, d, 71)
    sinks = torch.linspace(-2, 2, hkv * g, device=dev)
    rows, starts, firsts = list(range(6)), [2 * r for r in range(6)], [max(n - 2, 0) for n in lengths]
    counts = torch.tensor([min(n, 2) for n in lengths], dtype=torch.int32, device=dev)
    narrow = cache.tables
    for with_sinks in (None, sinks):
        lse, same = torch.empty(12, hkv * g, device=dev), torch.empty(12, hkv * g, device=dev)
        cache.tables = torch.cat([narrow, narrow[:, :1].expand(-1, 100 - narrow.shape[1])], 1).contiguous()
        out = cache.attend(q, rows, starts, firsts, 2, counts=counts, partitions=100, piece=16, sinks=with_sinks, lse=lse)
        fused = cache.attend(q, rows, starts, firsts, 2, counts=counts, partitions=100, piece=16, sinks=with_sinks, lse=same, fused=True)
        for r, n in enumerate(lengths):
            at = slice(2 * r, 2 * r + min(n, 2))
            assert torch.equal(out[at], fused[at]) and torch.equal(lse[at], same[at]), r
            if with_sinks is None:
                want, want_lse = cache.want(q[at], r, firsts[r], min(n, 2))
                close(out[at], want, msg=str(r))
                torch.testing.assert_close(lse[at].double().cpu(), want_lse, atol=1e-3, rtol=1e-4, msg=str(r))


@pytest.mark.parametrize("kind", ["bf16", "fp8"])
@pytest.mark.parametrize("rows", [43, 63, 64, 65, 127, 128, 129, 191, 255, 256, 257])
@pytest.mark.parametrize("alike", [False, True])
def test_every_row_has_its_place_in_the_list(kind, rows, alike):
    # more units than workgroups: rows are ranked by their last partitions, 64 a wavefront, up to 256; rows of one length
    # (ties), of none and of several partitions among them. Every row as in launches too small to be ranked
    lengths = [90 if alike else 1 + (37 * r) % 150 for r in range(6)]
    cache = Cache(kind, 3, 128, 128, 16, lengths, seed=rows)
    q = rand_q(rows, 12, 128, 72)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    of = [(5 * r + r // 6) % 6 for r in range(rows)]
    counts = [0 if r % 19 == 7 and not alike else 1 for r in range(rows)]
    def run(at, **kw):
        out = torch.zeros(rows, 12, 128, dtype=torch.bfloat16, device=dev)
        return cache.attend(q, [of[r] for r in at], list(at), [lengths[of[r]] - 1 for r in at], 1, counts=i32([counts[r] for r in at]),
                            out=out, partitions=3, piece=64, **kw)
    want = sum(run(range(r, min(r + 16, rows))).float() for r in range(0, rows, 16)).bfloat16()
    for fused in (False, True):
        assert torch.equal(run(range(rows), fused=fused), want)
    close(want[:1], cache.want(q[:1], of[0], lengths[of[0]] - 1, 1)[0])


def test_a_workspace_that_starts_on_any_float():
    pk = kernels()
    cache = Cache("int8", 2, 128, 128, 16, [900, 3000])
    q = rand_q(10, 8, 128, 65)
    want = cache.attend(q, [0, 1], [0, 5], [890, 2990], 5)
    floats = pk.workspace_floats(10, 8, 64, 128)
    for off in (1, 2, 3):
        ws = torch.empty(floats + 4, device=dev)[off:off + floats]
        assert torch.equal(cache.attend(q, [0, 1], [0, 5], [890, 2990], 5, partitions=64, workspace=ws), want), off


@pytest.mark.parametrize("d,hkv,g", [(128, 2, 4), (256, 2, 3)])
@pytest.mark.parametrize("page", [16, 48])
@pytest.mark.parametrize("position,count", [(0, 1), (0, 63), (1, 64), (63, 65), (127, 130), (500, 300)])
def test_prompt_chunks_at_the_edges_of_a_block_of_keys(d, hkv, g, page, position, count):
    pk = kernels()
    cache = Cache("bf16", hkv, d, d, page, [position + count, 40], seed=66)
    q = rand_q(count, hkv * g, d, 67).bfloat16()
    out = pk.prefill(q, cache.k, cache.v, "bf16", cache.tables[0], position, page)
    close(out, cache.want(q, 0, position, count)[0])


@pytest.mark.parametrize("n,k", [(9000, 700), (3000, 512), (50000, 2048)])
@pytest.mark.parametrize("equal", [1, 62, 63, 64, 65, 511, 512, 513, 600])
def test_picks_where_the_kth_score_has_many_near_it(n, k, equal):
    # `equal` scores tie at the k-th place (a list of up to 64 is ranked at once, longer ones go by digits), among neighbours
    # one bit apart, over a range of all signs or of fewer bits than the digit has
    g = torch.Generator().manual_seed(n + equal)
    wide = torch.randn(n, generator=g) * 10 ** torch.empty(n).uniform_(-3, 3, generator=g)
    near = (torch.randint(0, 1500, (n,), generator=g, dtype=torch.int32) + 0x40490000).view(torch.float32)
    for s in (wide, near):
        kth = s.sort(descending=True).values[k - 1].item()
        s = s.clone()
        s[torch.randperm(n, generator=g)[:equal]] = kth
        rows = torch.stack([s, -s, s.flip(0)]).to(dev)
        rows[2, ::50] = float("nan")
        ends = torch.tensor([n, n - 3, n], dtype=torch.int32, device=dev)
        want = torch.from_numpy(oracle_indexer.sparse_index(rows.double().cpu().numpy(), ends.cpu().numpy(), k))
        import crit_amd.sparse_indexer as si
        assert torch.equal(si.topk(rows, ends, k).long().cpu(), want)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("tokens,heads,d", [(18, 64, 128), (33, 16, 128), (4, 64, 128), (7, 16, 64), (11, 128, 128), (15, 64, 256)])
@pytest.mark.parametrize("n", [1, 12000, 12001, 16064, 64001])
def test_a_few_tokens_score_their_keys_together_as_alone(fp8, tokens, heads, d, n):
    # four to fifteen tokens share a workgroup's keys: edges of its steps of 64 keys, a last workgroup of one to three tokens
    import crit_amd.sparse_indexer as si
    g = torch.Generator().manual_seed(n + tokens)
    q = torch.randn(tokens, heads, d, generator=g).to(dev, torch.bfloat16)
    rows = torch.randn(n + 3, d, generator=g).to(dev, torch.bfloat16)
    keys, scales = (rows.to(torch.float8_e4m3fn), torch.rand(n + 3, generator=g).to(dev) + 0.5) if fp8 else (rows, None)
    w = torch.randn(tokens, heads, generator=g).to(dev)
    ends = torch.randint(0, n + 1, (tokens,), generator=g, dtype=torch.int32).to(dev)
    ends[0] = n
    slots = torch.randperm(n + 3, generator=g)[:n].int().to(dev)
    for kw in ({"slots": slots}, {"slots": slots[None]}, {}):
        got = si.scores(q, keys, w, ends, key_scales=scales, **kw)
        for t in (0, 1, 3, tokens - 1):
            alone = si.scores(q[t:t + 1], keys, w[t:t + 1], ends[t:t + 1], key_scales=scales, **kw)
            assert torch.equal(got[t], alone[0]), t


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("columns", [1, 2])
def test_latent_results_of_many_heads_in_rows_on_and_off_16_bytes(dtype, columns):
    import crit_amd.latent_attention as la
    g = torch.Generator().manual_seed(68)
    rows, page, lengths = 3, 64, [70, 1500, 33]
    tables = torch.randperm(100, generator=g).to(torch.int32)[:3 * 30].view(3, 30).to(dev)
    cache = torch.randn(100, page, 576, generator=g).to(dtype).to(dev)
    q = torch.randn(rows * columns, 128, 576, generator=g).to(dtype).to(dev)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    run = lambda **kw: la.attend(q, cache, tables, i32([0, 1, 2]), i32([columns * r for r in range(rows)]),
                                 torch.tensor([n - columns for n in lengths], device=dev), columns, page, rank=512, **kw)
    want = run()
    wide = torch.zeros(rows * columns, 128, 516, dtype=dtype, device=dev)      # rows of 1,032 bytes
    run(out=wide[:, :, :512])
    assert torch.equal(wide[:, :, :512], want) and not bool(wide[:, :, 512:].any())
    assert torch.equal(run(out=torch.empty(rows * columns, 128, 512, device=dev)).to(dtype), want)

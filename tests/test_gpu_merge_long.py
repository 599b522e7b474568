"""The merge of few rows of many partitions, a workgroup a share of the value dims: the fused launch's bits, at counts of
partitions around what a wavefront takes (32), a chunk of 256-wide values (128) and of narrower ones (256), several rows of
different lengths beside each other, with sinks and log-sum-exps. And the merge of more rows, whose lanes take a value's dims 64
apart."""
import pytest
import torch

from tests.support import Cache, rand_q

pytestmark = pytest.mark.gpu
dev = "cuda"


@pytest.mark.parametrize("kind", ["bf16", "fp8", "int8"])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_the_bits_of_the_fused_launch(kind, d, out_dtype):
    hq, hkv, piece = 4, 2, 64
    counts = [1, 32, 33, 36, 127, 128, 129, 256, 257, 259]
    lengths = [piece * n - (7 if n % 2 else 0) for n in counts]
    cache = Cache(kind, hkv, d, d, 16, lengths, seed=d)
    q = rand_q(len(counts), hq, d, 5).to(torch.bfloat16)
    sinks = torch.linspace(-2.0, 2.0, hq, device=dev)
    rows, firsts = list(range(len(counts))), [n - 1 for n in lengths]
    found = []
    for fused in (False, True):
        for sink in (None, sinks):
            lse = torch.full((len(counts), hq), 7.0, device=dev)
            out = torch.empty(len(counts), hq, d, dtype=out_dtype, device=dev)
            cache.attend(q, rows, rows, firsts, 1, fused=fused, partitions=300, piece=piece, sinks=sink, lse=lse, out=out)
            found.append((out, lse))
    for (a, b), (x, y) in zip(found[:2], found[2:]):
        assert torch.equal(a, x) and torch.equal(b, y)
    for i in (2, 6, 9):
        want, want_lse = cache.want(q[i:i + 1], i, firsts[i], 1)
        torch.testing.assert_close(found[0][0][i:i + 1].double().cpu(), want, atol=8e-3, rtol=2e-2)
        torch.testing.assert_close(found[0][1][i:i + 1].double().cpu(), want_lse, atol=1e-3, rtol=1e-4)


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [19, 20, 63])
def test_many_rows_of_different_lengths(rows, out_dtype):
    # 608, 640 and 2,016 triples of 1 to 40 partitions; results at an odd place of a wider tensor
    hq, hkv, d, piece = 32, 8, 128, 64
    counts = [1 + (7 * i) % 40 for i in range(rows)]
    lengths = [piece * n - (5 if n % 2 else 0) for n in counts]
    cache = Cache("bf16", hkv, d, d, 16, lengths, seed=rows)
    q = rand_q(rows, hq, d, 5).to(torch.bfloat16)
    sinks = torch.linspace(-2.0, 2.0, hq, device=dev)
    found = []
    for fused in (False, True):
        lse = torch.full((rows, hq), 7.0, device=dev)
        out = torch.empty(rows, hq, d + 3, dtype=out_dtype, device=dev)[..., 1:d + 1]
        cache.attend(q, list(range(rows)), list(range(rows)), [n - 1 for n in lengths], 1, fused=fused, partitions=40, piece=piece, sinks=sinks, lse=lse, out=out)
        found.append((out, lse))
    assert torch.equal(found[0][0], found[1][0]) and torch.equal(found[0][1], found[1][1])

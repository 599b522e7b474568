"""attend() and write() as an engine calls them, through the native host code: the bits of the same calls with the Python code alone,
over every page kind, on another stream, and from a graph. What the native code hands back is looked at, so that it is it that ran."""
import pytest
import torch

import crit_amd.paged_kv_attention as pk
from tests.support import Cache, bits, rand_q

pytestmark = pytest.mark.gpu
dev = "cuda"
KINDS = ["bf16", "fp16", "fp8", "fp8:row", "int8"]


class Spied:
    """The native host code, its answers kept."""

    def __init__(self, native):
        self.native, self.answers = native, []

    def attend(self, *given):
        self.answers.append(self.native.attend(*given))
        return self.answers[-1]

    def write(self, *given):
        self.answers.append(self.native.write(*given))
        return self.answers[-1]


@pytest.fixture
def spied(monkeypatch):
    assert pk._host is not None, "the native host code is not built"
    found = Spied(pk._host)
    monkeypatch.setattr(pk, "_host", found)
    return found


def calls(kind, form):
    """A window call of three uneven rows in one of its forms: (the call, into a result and log-sum-exps of its own, those)."""
    hq, hkv, d, columns, firsts = 8, 2, 128, 4, [700, 30, 1300]
    cache = Cache(kind, hkv, d, d, 16, [n + columns for n in firsts], seed=3)
    i32 = dict(dtype=torch.int32, device=dev)
    counts = [4, 2, 3] if form == "packed" else [columns] * 3
    starts = [0, counts[0], counts[0] + counts[1]]
    tokens = sum(counts)
    q = rand_q(tokens, hq, d, 5).to(dev, torch.float16 if kind == "fp16" else torch.bfloat16)
    given = dict(counts=torch.tensor(counts, **i32), offsets=torch.tensor(starts, **i32), tokens=tokens) if form == "packed" else {}
    if form == "tree":
        given["parents"] = torch.tensor([-1, 0, 0, 1] * 3, **i32)
    lse = torch.zeros(tokens, hq, device=dev) if form != "plain" else None
    out = torch.zeros(tokens, hq, d, dtype=q.dtype, device=dev)
    parts = pk.partitions(q.device, hkv, kind, d, d)
    work = torch.zeros(pk.workspace_floats(3 * columns, hq, parts, d), device=dev)
    fixed = [torch.arange(3, **i32), torch.tensor(starts, **i32), torch.tensor(firsts, dtype=torch.int64, device=dev)]

    def call():
        return pk.attend(q, cache.k, cache.v, kind, cache.tables, *fixed, columns, 16, key_scales=cache.ks, value_scales=cache.vs,
                         multipliers=cache.multipliers, partitions=parts, out=out, lse=lse, workspace=work, **given)
    return call, [out] if lse is None else [out, lse]


def by_python_alone(call, results, monkeypatch):
    with monkeypatch.context() as without:
        without.setattr(pk, "_host", None)
        call()
    want = [x.clone() for x in results]
    assert all(bool(x.any()) for x in want)
    for x in results:
        x.zero_()
    return want


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("form", ["plain", "lse", "packed", "tree"])
def test_a_windows_call_is_taken_natively_with_the_same_bits(kind, form, spied, monkeypatch):
    call, results = calls(kind, form)
    want = by_python_alone(call, results, monkeypatch)
    spied.answers.clear()      # (the cache was written through it)
    assert call() is results[0] and spied.answers == [0]
    for got, x in zip(results, want):
        assert torch.equal(got, x)


@pytest.mark.parametrize("kind", ["bf16", "fp8"])
def test_a_windows_call_on_another_stream_and_from_a_graph(kind, spied, monkeypatch):
    call, results = calls(kind, "packed")
    want = by_python_alone(call, results, monkeypatch)
    spied.answers.clear()
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        call()
    stream.synchronize()
    assert spied.answers == [0] and all(torch.equal(got, x) for got, x in zip(results, want))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    assert spied.answers == [0, 0]
    for _ in range(3):
        for x in results:
            x.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(got, x) for got, x in zip(results, want))
        call()      # (the program's own work between the replays)


def test_the_entrys_refusal_of_a_native_call_is_raised(spied):
    # the queries' strides are the library's to refuse: nothing is launched
    q = torch.zeros(1, 2, 132, dtype=torch.bfloat16, device=dev)[..., :128]
    pages = torch.zeros(2, 16, 2, 128, dtype=torch.bfloat16, device=dev)
    one = torch.zeros(1, dtype=torch.int32, device=dev)
    with pytest.raises(ValueError):
        pk.attend(q, pages, pages, "bf16", one[None], one, one, one.long(), 1, 16, partitions=8, out=torch.zeros(1, 2, 128, device=dev),
                  workspace=torch.zeros(pk.workspace_floats(1, 2, 8, 128), device=dev))
    assert len(spied.answers) == 1 and spied.answers[0] not in (None, 0)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("rotated", [False, True])
def test_an_append_is_taken_natively_with_the_same_bytes(kind, rotated, spied, monkeypatch):
    cache = Cache(kind, 2, 128, 128, 16, [40, 40], seed=1)
    g = torch.Generator().manual_seed(2)
    tokens = 37
    keys, values = (torch.randn(tokens, 2, 128, generator=g).to(dev, torch.bfloat16) for _ in range(2))
    rope = (torch.randn(64, 128, generator=g).to(dev), torch.randint(0, 64, (tokens,), generator=g).to(dev)) if rotated else None
    stores = [x for x in (cache.k, cache.v, cache.ks, cache.vs) if x is not None]
    before = [x.clone() for x in stores]
    slots = cache.slots(1, torch.arange(tokens, device=dev))

    def call():
        pk.write(keys, values, slots, cache.k, cache.v, kind, cache.ks, cache.vs, multipliers=cache.multipliers, rope=rope)
    with monkeypatch.context() as without:
        without.setattr(pk, "_host", None)
        call()
    want = [x.clone() for x in stores]
    for x, old in zip(stores, before):
        x.copy_(old)
    spied.answers.clear()
    call()
    assert spied.answers == [0]
    for got, x, old in zip(stores, want, before):
        assert torch.equal(bits(got), bits(x)) and not torch.equal(bits(got), bits(old))

"""The workloads the framework's speed is judged by: what an engine asks of it, over the range it asks it in.

A case is a plain dict: its "path" names the work, the rest its sizes and page kind.

    step      a decode step of a small batch: the step's buffers from the round tables, then for every layer the append
              of the new tokens (their keys rotated on the way in where "rope") and the attention over the pages
    append    the keys and values of a prompt (or of a few tokens) into one layer's pages
    decode    one layer's attention of a batch, a new token a sequence, over ragged contexts
    long      one layer's attention of a few very long sequences in contiguous splits, with the log-sum-exps
    verify    one layer's attention of a speculative round: several columns a sequence, as a chain or as a draft tree
    prefill   one layer's attention of prompt chunks on top of the prefixes already in the pages; "fresh": 8-bit pages
              with the chunk's own rows given unquantised beside them
    latent    one layer's multi-head latent attention of a batch over a cache of compressed rows
    index     sparse index selection: every token's k best keys by the indexer's scores

Pages are placed at random in a pool a quarter larger than what is used; queries, keys and values are normal, with one
value in a hundred twenty times as large where the pages are 8-bit (what makes the scales of such pages matter).
"""
import math

import torch

import crit_amd.latent_attention as la
import crit_amd.paged_kv_attention as pk
import crit_amd.sparse_indexer as si

STORE = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp8": torch.float8_e4m3fn, "fp8:row": torch.float8_e4m3fn,
         "int8": torch.int8}
RANK, ROPE = 512, 64        # a latent cache's row: the compressed part and the rotary key
LARGEST_BYTES = 2.4e9       # what the largest listed case reads: no drawn case reads more
LARGEST_FLOPS = 2.8e11      # ... or multiplies more


def listed():
    return [
        # An engine with a handful of users: launches and the host's calls between them count, not the bytes.
        dict(name="step_3rows_bf16", path="step", kind="bf16", hq=32, hkv=8, d=128, page=16, rows=3, lo=700, hi=4000,
             layers=8, rope=True),
        # A step's prompt tokens (8 chunks of 512 and 56 decode rows) go into the pages of a quantised cache.
        dict(name="append_4152tokens_fp8", path="append", kind="fp8", hq=32, hkv=8, d=128, page=16, rows=4152, rope=False),
        # A full batch of an 8B model, 16-bit cache: the benchmark's own workload, one layer of it.
        dict(name="decode_64rows_bf16", path="decode", kind="bf16", hq=32, hkv=8, d=128, page=16, rows=64, lo=1024, hi=8192),
        # The same model with an FP8 cache, twice the batch at twice the length: the largest.
        dict(name="decode_128rows_fp8", path="decode", kind="fp8", hq=32, hkv=8, d=128, page=16, rows=128, lo=2048, hi=16384),
        # A small batch of a model with wide heads and row-scaled pages of 64 positions.
        dict(name="decode_8rows_fp8row_x256", path="decode", kind="fp8:row", hq=24, hkv=4, d=256, page=64, rows=8, lo=15000, hi=16500),
        # One document of 200 thousand tokens.
        dict(name="long_1row_bf16", path="long", kind="bf16", hq=40, hkv=8, d=128, page=16, rows=1, lo=200000, hi=200000),
        # A full batch that verifies four drafted tokens and its own.
        dict(name="verify_64rows_5cols_bf16", path="verify", kind="bf16", hq=32, hkv=8, d=128, page=16, rows=64, lo=1024,
             hi=8192, columns=5, tree=False),
        # One long sequence that verifies a draft tree, INT8 pages.
        dict(name="verify_1row_8cols_int8", path="verify", kind="int8", hq=56, hkv=8, d=128, page=16, rows=1, lo=50000,
             hi=50000, columns=8, tree=True),
        # Chunked prefill of eight prompts at once, on prefixes of up to 8,192 positions.
        dict(name="prefill_8x512_bf16", path="prefill", kind="bf16", hq=32, hkv=8, d=128, page=16, rows=8, count=512, lo=0,
             hi=8192, fresh=False),
        # One ragged chunk of a model with wide heads after a short prefix.
        dict(name="prefill_777_bf16_x256", path="prefill", kind="bf16", hq=24, hkv=2, d=256, page=16, rows=1, count=777,
             lo=1024, hi=1024, fresh=False),
        # A full batch of a latent-attention model, every head on this GPU.
        dict(name="latent_64rows_128heads_bf16", path="latent", kind="bf16", hq=128, page=64, rows=64, lo=1024, hi=8192, columns=1),
        # A sparse-attention model's few tokens choose among the 50,000 keys they see.
        dict(name="index_4tokens_50000keys", path="index", kind="bf16", hq=64, d=128, rows=4, keys=50000, k=2048),
    ]


def _spread(rng, lo, hi):
    """A size within lo .. hi, spread over its logarithm, as odd as it comes."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _heads(rng, kind):
    """The models' head shapes: (query heads, KV heads, width, page)."""
    hq, hkv, d = rng.choice([(32, 8, 128), (32, 8, 128), (40, 8, 128), (56, 8, 128), (24, 4, 256), (24, 2, 256), (32, 8, 64)])
    return dict(kind=kind, hq=hq, hkv=hkv, d=d, page=rng.choice([16, 16, 64]))


def _fits(case):
    """No dearer than the largest listed case: several columns cost twice a column's bytes, other widths than 128 up to
    three times a 128-wide chunk's products."""
    w = work(case)
    most_bytes = LARGEST_BYTES / (2 if case["path"] == "verify" else 1)
    most_flops = LARGEST_FLOPS / (3 if case["path"] == "prefill" and case["d"] != 128 else 1)
    return w["bytes"] <= most_bytes and w["flops"] <= most_flops


def draw(rng):
    path = rng.choice(["step", "append", "decode", "decode", "long", "verify", "prefill", "latent", "index"])
    kind = rng.choice(["bf16", "bf16", "fp16", "fp8", "fp8", "fp8:row", "int8"])
    while True:
        if path == "step":
            hi = _spread(rng, 256, 8192)
            case = dict(path=path, **_heads(rng, kind), rows=_spread(rng, 1, 16), lo=max(1, hi // rng.choice([1, 2, 8])), hi=hi,
                        layers=rng.choice([4, 8]), rope=rng.random() < 0.5)
        elif path == "append":
            case = dict(path=path, **_heads(rng, kind), rows=_spread(rng, 1, 65536), rope=rng.random() < 0.3)
        elif path == "decode":
            hi = _spread(rng, 512, 16384)
            case = dict(path=path, **_heads(rng, kind), rows=_spread(rng, 1, 128), lo=max(1, hi // rng.choice([1, 2, 8])), hi=hi)
        elif path == "long":
            hi = _spread(rng, 32768, 200000)
            case = dict(path=path, **_heads(rng, kind), rows=rng.randint(1, 4), lo=hi, hi=hi)
        elif path == "verify":
            hi = _spread(rng, 512, 65536)
            case = dict(path=path, **_heads(rng, kind), rows=_spread(rng, 1, 64), lo=max(1, hi // rng.choice([1, 2, 8])), hi=hi,
                        columns=rng.randint(2, 8), tree=rng.random() < 0.3)
        elif path == "prefill":
            hi = _spread(rng, 256, 16384)
            heads = _heads(rng, "bf16" if kind == "fp16" else kind)
            if heads["d"] == 256 and kind == "int8":
                heads["kind"] = "fp8"
            case = dict(path=path, **heads, rows=rng.choice([1, 1, 2, 4, 8]), count=_spread(rng, 16, 2048),
                        lo=rng.choice([0, hi]), hi=hi, fresh=heads["kind"] != "bf16" and rng.random() < 0.3)
        elif path == "latent":
            hi = _spread(rng, 512, 16384)
            case = dict(path=path, kind=rng.choice(["bf16", "fp8"]), hq=rng.choice([16, 32, 64, 128, 128]), page=64,
                        rows=_spread(rng, 1, 64), lo=max(1, hi // rng.choice([1, 2, 8])), hi=hi, columns=rng.choice([1, 1, 2]))
        else:
            case = dict(path=path, kind=rng.choice(["bf16", "fp8"]), hq=64, d=128, rows=_spread(rng, 1, 1024),
                        keys=_spread(rng, 4096, 65536), k=rng.choice([512, 2048]))
        if _fits(case):
            return case


# -- sizes ---------------------------------------------------------------------------------------------------------------
def _contexts(case):
    """Every row's positions already in the pages, evenly over lo .. hi (which row has which is the seed's)."""
    n, lo, hi = case["rows"], case["lo"], case["hi"]
    return [lo + (hi - lo) * (2 * i + 1) // (2 * n) for i in range(n)]


def _item(kind):
    return 2 if kind in ("bf16", "fp16") else 1


def work(case):
    path, kind, e = case["path"], case["kind"], _item(case["kind"])
    if path == "index":
        tokens, n, h, d, k = case["rows"], case["keys"], case["hq"], case["d"], case["k"]
        seen = sum(_index_ends(case))
        return {"bytes": n * (d * e + (4 if e == 1 else 0)) + tokens * (h * d * 2 + h * 4 + k * 4), "flops": 2 * h * d * seen}
    if path == "latent":
        c, h = case["columns"], case["hq"]
        rows = sum(n + c for n in _contexts(case))
        seen = sum(n + j + 1 for n in _contexts(case) for j in range(c))
        row = (RANK + ROPE) * e + (8 if e == 1 else 0)
        return {"bytes": rows * row + case["rows"] * c * h * (2 * RANK + ROPE) * 2, "flops": 2 * h * (2 * RANK + ROPE) * seen}
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    row = 2 * hkv * (d * e + (4 if kind in ("fp8:row", "int8") else 0))      # a position's keys and values, with their scales
    if path == "append":
        return {"bytes": case["rows"] * (row + 2 * hkv * d * 2 + 8), "flops": 0}
    new = {"step": 1, "verify": case.get("columns", 1), "prefill": case.get("count", 1)}.get(path, 1)
    layers = case.get("layers", 1)
    total = sum(n + new for n in _contexts(case))
    seen = sum(n * new + new * (new + 1) // 2 for n in _contexts(case))
    tokens = case["rows"] * new
    moved = total * row + 2 * tokens * hq * d * 2
    if path == "step":
        moved += tokens * (row + 2 * hkv * d * 2)
    return {"bytes": layers * moved, "flops": layers * 4 * hq * d * seen}


def tolerance(case):
    """Attention: 16-bit probabilities and 16-bit results, measured against 64 bits at 1.7e-3 .. 2.4e-3 (largest 1.3e-2) with
    BF16 and 2.6e-4 (9e-4) with FP16. Bytes in the pages, slots and picks are whole numbers that do not change."""
    if case["path"] in ("append", "index"):
        return "exact"
    return {"rel": 1.2e-3, "max": 6e-3, "differ": 0.0} if case["kind"] == "fp16" else {"rel": 1e-2, "max": 0.06, "differ": 0.0}


# -- inputs --------------------------------------------------------------------------------------------------------------
def _normal(g, *shape, dtype=torch.bfloat16):
    return torch.randn(*shape, device="cuda", dtype=torch.bfloat16, generator=g).to(dtype)


def _values(g, shape, kind):
    """Keys or values as a projection gives them; one in a hundred large where the cache is 8-bit."""
    x = torch.randn(shape, device="cuda", dtype=torch.bfloat16, generator=g)
    if _item(kind) == 1:
        x *= torch.where(torch.rand(shape, device="cuda", dtype=torch.bfloat16, generator=g) < 0.01, 20.0, 1.0).to(torch.bfloat16)
    return x


def _stored(x, kind):
    """(pages, row scales or None, the heads' multipliers or None) of rows x [...][heads][d]."""
    if kind in ("bf16", "fp16"):
        return x.to(STORE[kind]), None, None
    if kind == "fp8":
        m = x.abs().amax(dim=tuple(range(x.dim() - 2)) + (x.dim() - 1,)).float() / 448.0
        return (x / m.to(torch.bfloat16)[:, None]).clamp(-448, 448).to(STORE[kind]), None, m
    top = 448.0 if kind == "fp8:row" else 127.0
    s = (x.abs().amax(dim=-1).float() / top).clamp(min=1e-30)
    y = (x / s[..., None].to(torch.bfloat16)).clamp(-top, top)
    return (y.round() if kind == "int8" else y).to(STORE[kind]), s, None


class _Pool:
    """One layer's pages for rows of the given lengths (every row's positions, the new ones among them), random places."""

    def __init__(self, case, lengths, g, cpu, tables=None):
        kind, hkv, d, page = case["kind"], case["hkv"], case["d"], case["page"]
        pages = [-(-n // page) for n in lengths]
        n_pages = sum(pages) * 5 // 4 + 1
        if tables is None:
            tables = torch.full((len(pages), -(-max(pages) // 16) * 16), n_pages, dtype=torch.int32)      # unused: the dump page
            order, at = torch.randperm(n_pages, generator=cpu).to(torch.int32), 0
            for r, w in enumerate(pages):
                tables[r, :w] = order[at:at + w]
                at += w
            tables = tables.cuda()
        self.tables, self.dump = tables, n_pages
        shape = (n_pages + 1, page, hkv, d)
        self.k, self.ks, km = _stored(_values(g, shape, kind), kind)
        self.v, self.vs, vm = _stored(_values(g, shape, kind), kind)
        self.multipliers = torch.stack([km, vm]).contiguous() if km is not None else (1.0, 1.0)
        self.scales = dict(key_scales=self.ks, value_scales=self.vs, multipliers=self.multipliers)
        raw = lambda x: x.view(torch.uint8) if x.dtype == STORE["fp8"] else x
        self.state = [raw(x) for x in (self.k, self.v, self.ks, self.vs) if x is not None]


def _index_ends(case):
    """The keys a token sees: the last tokens of a prompt, one more each."""
    return [max(1, case["keys"] - case["rows"] + t + 1) for t in range(case["rows"])]


def _rope_table(d):
    angle = torch.arange(16384, dtype=torch.float32, device="cuda")[:, None] / \
        (10000.0 ** (torch.arange(d // 2, dtype=torch.float32, device="cuda") / (d // 2)))[None, :]
    return torch.cat([angle.cos(), angle.sin()], 1).contiguous()


def prepare(case, seed):
    g, cpu = torch.Generator(device="cuda").manual_seed(seed), torch.Generator().manual_seed(seed)
    path, kind = case["path"], case["kind"]
    rows = case["rows"]
    s = {"case": case}
    if path == "index":
        d, n, h = case["d"], case["keys"], case["hq"]
        keys = _normal(g, n, d)
        if kind == "fp8":
            s["key_scales"] = keys.abs().amax(dim=-1).float() / 448.0
            keys = (keys / s["key_scales"][:, None].to(torch.bfloat16)).clamp(-448, 448).to(STORE["fp8"])
        s.update(q=_normal(g, rows, h, d), keys=keys, weights=torch.rand(rows, h, device="cuda", generator=g),
                 ends=torch.tensor(_index_ends(case), dtype=torch.int32).cuda(),
                 out=torch.empty(rows, case["k"], dtype=torch.int32, device="cuda"))
        return s
    if path == "append":
        hkv, d, page = case["hkv"], case["d"], case["page"]
        pool = _Pool(case, [rows], g, cpu)
        positions = torch.arange(rows, device="cuda")
        s.update(pool=pool, keys=_values(g, (rows, hkv, d), kind), values=_values(g, (rows, hkv, d), kind), positions=positions,
                 slots=pool.tables[0].long()[positions // page] * page + positions % page, rope=_rope_table(d) if case["rope"] else None)
        return s
    contexts = torch.tensor(_contexts(case))[torch.randperm(rows, generator=cpu)].tolist()
    new = {"step": 1, "verify": case.get("columns", 1), "prefill": case.get("count", 1), "latent": case.get("columns", 1)}.get(path, 1)
    lengths = [n + new for n in contexts]
    tokens = rows * new
    each = dict(dtype=torch.int32, device="cuda")
    s["firsts"] = torch.tensor(contexts, dtype=torch.int64).cuda()
    s["rows"], s["counts"] = torch.arange(rows, **each), torch.full((rows,), new, **each)
    s["starts"] = torch.arange(0, tokens, new, **each)
    if path == "latent":
        page, width = case["page"], RANK + ROPE
        pages = [-(-n // page) for n in lengths]
        n_pages = sum(pages) * 5 // 4 + 1
        tables, order, at = torch.zeros(rows, max(pages), dtype=torch.int32), torch.randperm(n_pages, generator=cpu).to(torch.int32), 0
        for r, w in enumerate(pages):
            tables[r, :w] = order[at:at + w]
            at += w
        cache = _normal(g, n_pages, page, width)
        if kind == "fp8":
            parts = cache.split([RANK, ROPE], dim=-1)
            s["scales"] = torch.stack([p.abs().amax(dim=-1).float() / 448.0 for p in parts], dim=-1).contiguous()
            cache = torch.cat([(p / s["scales"][..., i:i + 1].to(torch.bfloat16)).clamp(-448, 448) for i, p in enumerate(parts)], -1)
        s.update(cache=cache.to(STORE[kind]), tables=tables.cuda(), q=_normal(g, tokens, case["hq"], width),
                 out=torch.empty(tokens, case["hq"], RANK, dtype=torch.bfloat16, device="cuda"))
        return s
    hq, hkv, d, page = case["hq"], case["hkv"], case["d"], case["page"]
    kv16 = torch.float16 if kind == "fp16" else torch.bfloat16
    parts = pk.partitions(torch.device("cuda", torch.cuda.current_device()), hkv, kind, d, d)
    s["parts"] = parts
    if path == "step":
        layers = case["layers"]
        s["pools"] = [_Pool(case, lengths, g, cpu)]
        for _ in range(layers - 1):
            s["pools"].append(_Pool(case, lengths, g, cpu, s["pools"][0].tables))
        tables = s["pools"][0].tables
        s["buffers"] = pk.StepBuffers(rows, rows, tables.shape[1], s["pools"][0].dump, tables.device)
        s["capacity"] = torch.tensor([-(-n // page) * page for n in lengths], dtype=torch.int64).cuda()
        s["slot"] = torch.arange(rows, device="cuda")
        s["q"] = [_normal(g, rows, hq, d, dtype=kv16) for _ in range(layers)]
        s["keys"] = [_values(g, (rows, hkv, d), kind) for _ in range(layers)]
        s["values"] = [_values(g, (rows, hkv, d), kind) for _ in range(layers)]
        s["out"] = [torch.empty_like(q) for q in s["q"]]
        s["rope"] = _rope_table(d) if case["rope"] else None
        s["workspace"] = torch.empty(pk.workspace_floats(rows, hq, parts, d), dtype=torch.float32, device="cuda")
        return s
    s["pool"] = _Pool(case, lengths, g, cpu)
    s["q"] = _normal(g, tokens, hq, d, dtype=kv16)
    s["out"] = torch.empty_like(s["q"])
    if path == "prefill":
        if case["fresh"]:
            s["fresh"] = (_normal(g, tokens, hkv, d), _normal(g, tokens, hkv, d))
        s["position"] = contexts[0]
        return s
    if path == "long":
        s["lse"] = torch.empty(tokens, hq, dtype=torch.float32, device="cuda")
        s["chunk"] = pk.flash_chunk(d, d, hq, hkv, page, kind)
        parts = pk.flash_parts(s["pool"].tables.shape[1] * page, s["chunk"])
    if path == "verify" and case["tree"]:      # every node hangs from one of the two before it
        links = [[c - 1 if c < 2 or torch.rand((), generator=cpu) < 0.5 else c - 2 for c in range(new)] for _ in range(rows)]
        s["parents"] = torch.tensor(links, dtype=torch.int32).reshape(-1).cuda()
    s["workspace"] = torch.empty(pk.workspace_floats(tokens, hq, parts, d), dtype=torch.float32, device="cuda")
    return s


# -- one pass --------------------------------------------------------------------------------------------------------------
def run(s):
    case = s["case"]
    path, kind = case["path"], case["kind"]
    if path == "index":
        return si.select(s["q"], s["keys"], s["weights"], s["ends"], case["k"], key_scales=s.get("key_scales"), out=s["out"])
    if path == "latent":
        return la.attend(s["q"], s["cache"], s["tables"], s["rows"], s["starts"], s["firsts"], case["columns"], case["page"],
                         rank=RANK, counts=s["counts"], scales=s.get("scales"), out=s["out"])
    page = case["page"]
    if path == "append":
        pool = s["pool"]
        rope = None if s["rope"] is None else (s["rope"], s["positions"])
        pk.write(s["keys"], s["values"], s["slots"], pool.k, pool.v, kind, pool.ks, pool.vs, pool.multipliers, rope=rope)
        return pool.state
    if path == "step":
        pools = s["pools"]
        b = pk.step_buffers(s["buffers"], pools[0].tables, s["capacity"], s["firsts"], s["slot"], page, 8)
        rope = None if s["rope"] is None else (s["rope"], b.positions_t)
        for i, pool in enumerate(pools):
            pk.write(s["keys"][i], s["values"][i], b.d_slots, pool.k, pool.v, kind, pool.ks, pool.vs, pool.multipliers, rope=rope)
            pk.attend(s["q"][i], pool.k, pool.v, kind, b.d_tables, b.d_rows, b.d_starts, b.d_firsts, 1, page, counts=b.d_counts,
                      offsets=b.d_offsets, tokens=case["rows"], partitions=s["parts"], out=s["out"][i], workspace=s["workspace"],
                      **pool.scales)
        return {"out": s["out"], "slots": b.d_slots, "pages": [x for pool in pools for x in pool.state[:2]]}
    pool = s["pool"]
    if path == "prefill":
        if case["rows"] == 1:
            return pk.prefill(s["q"], pool.k, pool.v, kind, pool.tables[0], s["position"], page, out=s["out"], fresh=s.get("fresh"),
                              **pool.scales)
        return pk.prefill_rows(s["q"], pool.k, pool.v, kind, pool.tables, s["rows"], s["starts"], s["counts"], s["firsts"],
                               case["count"], page, out=s["out"], fresh=s.get("fresh"), **pool.scales)
    columns = case.get("columns", 1)
    if path == "long":
        out = pk.attend(s["q"], pool.k, pool.v, kind, pool.tables, s["rows"], s["starts"], s["firsts"], columns, page,
                        counts=s["counts"], flash=True, chunk=s["chunk"], out=s["out"], lse=s["lse"], workspace=s["workspace"],
                        **pool.scales)
        return out, s["lse"]
    return pk.attend(s["q"], pool.k, pool.v, kind, pool.tables, s["rows"], s["starts"], s["firsts"], columns, page,
                     counts=s["counts"], offsets=s["starts"], tokens=s["q"].shape[0], partitions=s["parts"],
                     parents=s.get("parents"), out=s["out"], workspace=s["workspace"], **pool.scales)


# -- the same in 64 bits -----------------------------------------------------------------------------------------------------
def _exact_rows(case, q, pool, firsts, scale, parents=None, fresh=None):
    """(out, log-sum-exps) of every row's window over its pages: q [rows][new][heads][dim], float64 on the GPU."""
    n_rows, new, hq, d = q.shape
    page, hkv = case["page"], case["hkv"]
    g = hq // hkv
    out, lse = torch.empty(n_rows, new, hq, d, dtype=torch.float64, device="cuda"), torch.empty(n_rows, new, hq, dtype=torch.float64, device="cuda")

    def real(x, scales, which, at, head):
        y = x.reshape(-1, hkv, d)[at, head].double()
        if scales is not None:
            y = y * scales.reshape(-1, hkv)[at, head].double()[:, None]
        if torch.is_tensor(pool.multipliers):
            y = y * pool.multipliers[which, head].double()
        return y

    for r in range(n_rows):
        first = firsts[r]
        n = torch.arange(first + new, device="cuda")
        at = pool.tables[r].long()[n // page] * page + n % page
        seen = torch.ones(new, first + new, dtype=torch.bool, device="cuda").tril(first)
        if parents is not None:      # of the window's own positions only a node's ancestors and itself
            for c in range(new):
                up, mine = c, []
                while up >= 0:
                    mine.append(up)
                    up = parents[r][up]
                seen[c, first:] = False
                seen[c, [first + m for m in mine]] = True
        for h in range(hkv):
            k, v = real(pool.k, pool.ks, 0, at, h), real(pool.v, pool.vs, 1, at, h)
            if fresh is not None:      # the chunk's own rows, unquantised
                k[first:], v[first:] = fresh[0][r, :, h].double(), fresh[1][r, :, h].double()
            x = q[r, :, h * g:(h + 1) * g].double().reshape(new * g, d) @ k.T.contiguous()
            x = (x * scale).reshape(new, g, -1).masked_fill(~seen[:, None, :], -math.inf)
            lse[r, :, h * g:(h + 1) * g] = x.logsumexp(-1)
            out[r, :, h * g:(h + 1) * g] = (x.softmax(-1).reshape(new * g, -1) @ v).reshape(new, g, d)
    return out, lse


def _coded(x, kind, pool, which):
    """A step's new rows as its pages hold them: (stored, row scales or None)."""
    x = x.float()
    if kind in ("bf16", "fp16"):
        return x.to(STORE[kind]), None
    if kind == "fp8":
        return (x / pool.multipliers[which][None, :, None]).clamp(-448, 448).to(STORE[kind]), None
    top = 448.0 if kind == "fp8:row" else 127.0
    s = (x.abs().amax(dim=-1) / top).clamp(min=1e-30)
    y = (x / s[..., None]).clamp(-top, top)
    return (y.round() if kind == "int8" else y).to(STORE[kind]), s


def _rotated(x, table, positions):
    """Keys turned by their positions' angles, pairs (j, j + dim / 2), rounded to their own type."""
    half = x.shape[-1] // 2
    row = table[positions][:, None, :]
    cos, sin, a, b = row[..., :half], row[..., half:], x[..., :half].float(), x[..., half:].float()
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1).to(x.dtype)


def exact(case, seed):
    """What run() returns, in 64 bits by plain torch; pages, slots and picks have no such value."""
    path, kind, rows = case["path"], case["kind"], case["rows"]
    if path in ("append", "index"):
        return None
    s = prepare(case, seed)
    firsts = s["firsts"].tolist()
    if path == "latent":
        new, page, h = case["columns"], case["page"], case["hq"]
        out = torch.empty(rows, new, h, RANK, dtype=torch.float64, device="cuda")
        q = s["q"].reshape(rows, new, h, RANK + ROPE)
        for r, first in enumerate(firsts):
            n = torch.arange(first + new, device="cuda")
            at = s["tables"][r].long()[n // page] * page + n % page
            kv = s["cache"].reshape(-1, RANK + ROPE)[at].double()
            if kind == "fp8":
                scales = s["scales"].reshape(-1, 2)[at].double()
                kv[:, :RANK] *= scales[:, :1]
                kv[:, RANK:] *= scales[:, 1:]
            for c in range(new):
                x = q[r, c].double() @ kv[:first + c + 1].T.contiguous() * (RANK + ROPE) ** -0.5
                out[r, c] = x.softmax(-1) @ kv[:first + c + 1, :RANK].contiguous()
        return out.reshape(rows * new, h, RANK)
    d, hq, page = case["d"], case["hq"], case["page"]
    if path == "step":
        outs = []
        for i, pool in enumerate(s["pools"]):
            keys = s["keys"][i] if s["rope"] is None else _rotated(s["keys"][i], s["rope"], s["firsts"])
            at = pool.tables.long()[torch.arange(rows, device="cuda"), s["firsts"] // page] * page + s["firsts"] % page
            for x, scales, new, which in ((pool.k, pool.ks, keys, 0), (pool.v, pool.vs, s["values"][i], 1)):
                codes, own = _coded(new, kind, pool, which)
                x.reshape(-1, case["hkv"], d)[at] = codes
                if own is not None:
                    scales.reshape(-1, case["hkv"])[at] = own
            outs.append(_exact_rows(case, s["q"][i][:, None], pool, firsts, d ** -0.5)[0][:, 0])
        return {"out": outs, "slots": None, "pages": [None] * (2 * len(outs))}
    tokens, new = s["q"].shape[0], s["q"].shape[0] // rows
    parents = s["parents"].reshape(rows, new).tolist() if "parents" in s else None
    fresh = [x.reshape(rows, new, case["hkv"], d) for x in s["fresh"]] if "fresh" in s else None
    out, lse = _exact_rows(case, s["q"].reshape(rows, new, hq, d), s["pool"], firsts, d ** -0.5, parents, fresh)
    out, lse = out.reshape(tokens, hq, d), lse.reshape(tokens, hq)
    return (out, lse) if path == "long" else out

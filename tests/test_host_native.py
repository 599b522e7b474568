"""The native share of attend()'s and write()'s host code: the parameters it fills are, byte for byte, the ones the Python code
fills, over the forms it takes; what it does not take (every mistake among it) it leaves to the Python code. On the CPU: with
no entry point to call it hands back the parameters."""
import ctypes
import itertools
import os

import pytest
import torch

import crit_amd.paged_kv_attention as pk
from crit_amd import build as builder

STORE = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp8": torch.float8_e4m3fn, "fp8:row": torch.float8_e4m3fn, "int8": torch.int8}
native = pytest.mark.skipif(pk._host is None, reason="the extension is not built")


def test_an_extension_that_is_built_is_in_use():
    # (one that does not load, or was built against something else, would leave the calls to the Python code without a word)
    if not os.path.exists(builder.HOST_LIB):
        pytest.skip("the extension is not built")
    assert pk._host is not None and os.path.samefile(pk._host.__file__, builder.HOST_LIB)


@pytest.fixture
def filled(monkeypatch):
    """The parameters of the general way's launch."""
    found = []
    monkeypatch.setattr(pk, "_require_device", lambda t, what: None)
    monkeypatch.setattr(pk, "_stream_of", lambda device: 0)
    monkeypatch.setattr(pk, "_launch_state", lambda device, stream: 0x1000)
    monkeypatch.setattr(pk, "_launch", lambda device, name, what, p, stream=None: found.append(bytes(p)))
    return found


def window(kind, hq=8, hkv=2, d=128, dv=128, page=16, rows=3, columns=2, rows_dtype=torch.int32, links=None, packed=True,
           per_head=False, lse=True, out_dtype=None, scale=None):
    t16 = torch.float16 if kind == "fp16" else torch.bfloat16
    tokens = rows * columns
    i32 = dict(dtype=torch.int32)
    scaled = kind in ("fp8:row", "int8")
    # (a slice of a wider projection, a slice of wider tables: the strides are the call's)
    return dict(q=torch.zeros(tokens, 3 * hq, d, dtype=t16)[:, hq:2 * hq], key_pages=torch.zeros(6, page, hkv, d, dtype=STORE[kind]),
                value_pages=torch.zeros(6, page, hkv, dv, dtype=STORE[kind]), kind=kind, tables=torch.zeros(4, 9, **i32)[:, :5],
                rows=torch.zeros(rows, dtype=rows_dtype), starts=torch.zeros(rows, **i32), firsts=torch.zeros(rows, dtype=torch.int64),
                columns=columns, page=page, counts=torch.zeros(rows, **i32) if packed else None,
                offsets=torch.zeros(rows, **i32) if packed else None, tokens=tokens if packed else None,
                key_scales=torch.zeros(6, page, hkv) if scaled else None, value_scales=torch.zeros(6, page, hkv) if scaled else None,
                multipliers=torch.ones(2, hkv) if per_head else (0.5, 0.25), scale=scale, partitions=64,
                parents=None if links is None else torch.zeros(tokens, dtype=links),
                out=torch.zeros(tokens, 2 * hq, dv, dtype=out_dtype or t16)[:, :hq], lse=torch.zeros(tokens, hq) if lse else None,
                workspace=torch.zeros(pk.workspace_floats(tokens, hq, 64, dv)))


ORDER = ("q", "key_pages", "value_pages", "tables", "rows", "starts", "firsts", "columns", "page", "counts", "offsets", "tokens",
         "key_scales", "value_scales", "multipliers", "scale", "partitions", "parents", "out", "lse", "workspace")


def attend_native(case):
    return pk._host.attend(0, 0, 0x1000, pk.KINDS[case["kind"]], case["kind"] == "fp16", *[case[name] for name in ORDER])


@native
@pytest.mark.parametrize("kind", list(STORE))
def test_a_windows_parameters_are_the_general_ways(kind, filled):
    forms = [dict(d=d, dv=dv) for d, dv in itertools.product(pk.HEAD_WIDTHS, pk.HEAD_WIDTHS)]
    forms += [dict(rows_dtype=torch.int64), dict(links=torch.int32), dict(links=torch.int64), dict(packed=False), dict(per_head=True), dict(lse=False),
              dict(out_dtype=torch.float32), dict(scale=0.3), dict(scale=-1.5), dict(hq=7, hkv=7, rows=1, columns=64), dict(page=24)]
    for form in forms:
        case = window(kind, **form)
        got = attend_native(case)
        pk.attend(**case)
        assert got is not None and got == filled[-1], form


@native
def test_other_forms_of_a_window_and_every_mistake_are_left_alone():
    case = window("bf16")
    assert attend_native(case) is not None
    class Own(torch.Tensor):
        pass
    wrong = dict(q=[case["q"].float(), case["q"][0], case["q"].transpose(1, 2), case["q"].as_subclass(Own), None],
                 key_pages=[case["key_pages"].half(), case["key_pages"][..., :64], None], value_pages=[None, torch.zeros(6, 16, 2, 96, dtype=torch.bfloat16)],
                 tables=[case["tables"].long(), case["tables"].t(), case["tables"][0]], rows=[case["rows"].short()],
                 starts=[case["starts"].long(), case["starts"][:0]], firsts=[case["firsts"].int()], columns=[0, 65, 2.0, True], page=[0, None],
                 counts=[case["counts"].long()], offsets=[None, case["offsets"].long()], tokens=[None, 2.0],
                 key_scales=[torch.zeros(6, 16, 2)], multipliers=[(1.0,), torch.ones(2, 3), torch.ones(2, 2).half(), [1.0, 1.0], (1, 1)],
                 scale=["1"], partitions=[None, 0], parents=[case["rows"][:2], torch.zeros(6), torch.zeros(6, 1, dtype=torch.int32)],
                 out=[torch.zeros(6, 8, 64), torch.zeros(6, 8, 128, dtype=torch.float64), torch.zeros(6, 8, 128).transpose(1, 2)],
                 lse=[torch.zeros(6, 8).half(), torch.zeros(6, 16)[:, ::2]], workspace=[case["workspace"][:-1], case["workspace"][::2], case["workspace"].half()])
    for name, values in wrong.items():
        for value in values:
            assert attend_native({**case, name: value}) is None, (name, value)
    for kind in ("fp8:row", "int8"):
        scaled = window(kind)
        assert attend_native({**scaled, "key_scales": None}) is None and attend_native({**scaled, "value_scales": None}) is None
    assert attend_native({**window("bf16", columns=65, rows=1), "parents": None}) is None
    # more partials than 64 bits count: no workspace holds them (a count that wraps would be below any)
    for heads, tokens, partitions in ((128, 1 << 40, 1 << 15), (128, (1 << 40) - 1, 65535), (8, 1 << 40, (1 << 31) - 1)):
        case_of = window("bf16", hq=heads, hkv=2)
        assert attend_native(case_of) is not None
        assert attend_native({**case_of, "tokens": tokens, "partitions": partitions}) is None, (heads, tokens, partitions)
    # a batch of calls under a transform is not one call
    from torch._C._functorch import _add_batch_dim, _vmap_decrement_nesting, _vmap_increment_nesting
    level = _vmap_increment_nesting(2, "error")
    try:
        assert attend_native({**case, "q": _add_batch_dim(torch.zeros(2, *case["q"].shape, dtype=torch.bfloat16), 0, level)}) is None
    finally:
        _vmap_decrement_nesting()


def rows(kind, hkv=2, d=128, dv=128, dtype=torch.bfloat16, rope=False, per_head=False, tokens=5):
    scaled = kind in ("fp8:row", "int8")
    return dict(keys=torch.zeros(tokens, 3 * hkv, d, dtype=dtype)[:, hkv:2 * hkv], values=torch.zeros(tokens, hkv, dv, dtype=dtype),
                slots=torch.zeros(tokens, dtype=torch.int64), key_pages=torch.zeros(4, 16, hkv, d, dtype=STORE[kind]),
                value_pages=torch.zeros(4, 16, hkv, dv, dtype=STORE[kind]), kind=kind, key_scales=torch.zeros(4, 16, hkv) if scaled else None,
                value_scales=torch.zeros(4, 16, hkv) if scaled else None, multipliers=torch.ones(2, hkv) if per_head else (0.5, 0.25),
                rope=(torch.zeros(7, d), torch.zeros(tokens, dtype=torch.int64)) if rope else None)


def write_native(case):
    return pk._host.write(0, 0, pk.KINDS[case["kind"]], case["kind"] == "fp16", case["keys"], case["values"], case["slots"], case["key_pages"],
                          case["value_pages"], case["key_scales"], case["value_scales"], case["multipliers"], case["rope"])


@native
@pytest.mark.parametrize("kind", list(STORE))
def test_an_appends_parameters_are_the_general_ways(kind, filled):
    forms = [dict(d=d, dv=dv, dtype=dtype) for d, dv, dtype in itertools.product((64, 128, 192), (64, 256), (torch.float32, torch.float16, torch.bfloat16))]
    forms += [dict(rope=True), dict(rope=True, d=256, dv=64), dict(per_head=True), dict(hkv=1, tokens=1)]
    for form in forms:
        case = rows(kind, **form)
        got = write_native(case)
        pk.write(**case)
        assert got is not None and got == filled[-1], form
    assert ctypes.sizeof(pk._abi.WriteParams) == len(filled[-1])


@native
def test_other_forms_of_an_append_and_every_mistake_are_left_alone():
    case = rows("bf16", rope=True)
    assert write_native(case) is not None
    table, positions = case["rope"]
    wrong = dict(keys=[case["keys"].double(), case["keys"].transpose(0, 2), case["keys"][:0], case["keys"].float(), None],
                 values=[None, case["values"].float(), torch.zeros(5, 2, 256, dtype=torch.bfloat16)], slots=[case["slots"].int(), torch.zeros(10, dtype=torch.int64)[::2]],
                 key_pages=[None, case["key_pages"].half(), case["key_pages"].transpose(0, 1)], value_pages=[None, case["value_pages"].transpose(0, 1)],
                 key_scales=[torch.zeros(4, 16, 2)], multipliers=[None, (1.0, 1), torch.ones(2, 4)[:, ::2]],
                 rope=[(table,), (table, positions, "half"), (table, positions, "interleaved", 1.0), (table.half(), positions), (table[:, :64], positions),
                       (table[:0], positions), (table, positions.int()), (table, positions[:4]), [table, positions]])
    for name, values in wrong.items():
        for value in values:
            assert write_native({**case, name: value}) is None, (name, value)
    assert write_native({**rows("int8"), "key_scales": None}) is None and write_native({**rows("int8"), "value_scales": None}) is None
    assert write_native(rows("bf16", d=192, rope=True)) is None

"""The native call module and ops.py's own path give the same results, errors and refusals."""

from __future__ import annotations

import pytest
import torch

from attnarc_amd import _native, ops, workloads

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class _NoCalls:
    """Stands in for the call module and takes no call."""

    def decode_extended(self, *args):
        return None

    decode_views = rope_write = decode_extended


def _both(monkeypatch, call):
    """call() through the native module and through ops.py; each its value or its error."""
    got = []
    for module in (_native.calls(), _NoCalls()):
        monkeypatch.setattr(_native, "_calls", module)
        try:
            got.append(call())
        except Exception as e:  # noqa: BLE001
            got.append((type(e), str(e)))
        monkeypatch.undo()
    torch.cuda.synchronize()
    return got


def _case(kv="native", partition=0, layout="NHD", dtype=torch.bfloat16, per_head=True):
    return workloads.make_case(
        name="calls", dtype=dtype, sequences=3, query_heads=8, kv_heads=2, head_size=64, value_head_size=64,
        block_size=16, lengths=[1, 70, 301], seed=5, device=DEV, cache_encoding=kv, layout=layout,
        partition_tokens=partition, per_head_scales=per_head)


def _extended(c, **kw):
    args = dict(max_sequence_length=c.max_sequence_length, scale=c.scale, layout=c.layout, key_scales=c.key_scales,
                value_scales=c.value_scales, partition_tokens=c.partition_tokens)
    args.update(kw)
    return ops.paged_decode_attention_extended(c.query, c.key_cache, c.value_cache, c.block_tables,
                                               c.sequence_lengths, **args)


@pytest.mark.parametrize("kv,partition,layout,dtype,per_head", [
    ("native", 0, "NHD", torch.float32, True), ("native", 64, "HND", torch.float16, True),
    ("fp8", 128, "HND", torch.bfloat16, True), ("fp8", 0, "NHD", torch.float16, False)])
@pytest.mark.parametrize("own", ["nothing", "output", "output and lse", "workspace"])
def test_extended_calls_agree(monkeypatch, kv, partition, layout, dtype, per_head, own):
    c = _case(kv, partition, layout, dtype, per_head)
    kw = {"scale": None, "return_lse": True}
    if own.startswith("output"):
        kw["output"] = torch.empty_like(c.query)
    if own == "output and lse":
        kw["lse"] = torch.empty(c.query.shape[:2], device=DEV)
    if own == "workspace" and partition:
        need = ops.extended_workspace_elements(3, 8, 64, c.max_sequence_length, partition)
        kw["workspace"] = torch.empty(need + 5, device=DEV)
    (out, lse), (want, want_lse) = _both(monkeypatch, lambda: [x.clone() for x in _extended(c, **kw)])
    assert torch.equal(out, want) and torch.equal(lse, want_lse) and out.dtype == dtype
    if "output" in kw:
        assert _extended(c, **kw)[0] is kw["output"]


@pytest.mark.parametrize("what", [
    "layout", "scale", "length", "negative length", "float length", "workspace", "requires grad", "cpu tables",
    "strided query", "scales missing", "dtype", "table type", "no tokens", "big partition"])
def test_refusals_agree(monkeypatch, what):
    c = _case("fp8" if what == "scales missing" else "native", 64)
    kw = {}
    if what == "layout":
        kw["layout"] = "NDH"
    if what == "scale":
        kw["scale"] = -1.0
    if what == "length":
        kw["max_sequence_length"] = 100000
    if what == "negative length":
        kw["max_sequence_length"] = -1
    if what == "float length":
        kw["max_sequence_length"] = 301.0
    if what == "workspace":
        kw["workspace"] = torch.empty(3, device=DEV)
    if what == "requires grad":
        c.query = c.query.requires_grad_()
    if what == "cpu tables":
        c.query = c.query.cpu()  # refused before anything is read
        kw["layout"] = "NDH"
    if what == "strided query":
        c.query = c.query.transpose(0, 1).contiguous().transpose(0, 1)
    if what == "scales missing":
        kw["key_scales"] = None
    if what == "dtype":
        c.key_cache = c.key_cache.half()
    if what == "table type":
        c.block_tables = c.block_tables.long()
    if what == "no tokens":
        kw["max_sequence_length"] = 0
    if what == "big partition":
        kw["partition_tokens"] = 1 << 32
    a, b = _both(monkeypatch, lambda: _extended(c, **kw))
    if what == "float length":
        assert torch.equal(a, b)
    else:
        assert isinstance(a, tuple) and a == b


def test_base_operator_and_write_agree(monkeypatch):
    c = _case()

    def base(length=c.max_sequence_length, tables=c.block_tables):
        return ops.paged_decode_attention(c.query, c.key_cache, c.value_cache, tables, c.sequence_lengths,
                                          max_sequence_length=length)

    a, b = _both(monkeypatch, base)
    assert torch.equal(a, b)
    for bad in (lambda: base(1 << 40), lambda: base(0), lambda: base(tables=c.block_tables.long())):
        a, b = _both(monkeypatch, bad)
        assert isinstance(a, tuple) and a == b

    def write(kv="fp8", neox=True, **swap):
        w = workloads.rope_write_case(9, DEV, cache_encoding=kv)
        args = dict(query=w.query, key=w.key, value=w.value, positions=w.positions, cos_sin_cache=w.cos_sin_cache,
                    kv_cache=w.kv_cache, key_scales=w.key_scales, value_scales=w.value_scales,
                    slot_mapping=w.slot_mapping)
        args.update({k: f(args[k]) for k, f in swap.items()})
        return [t.clone() for t in ops.rope_paged_kv_write_(*args.values(), neox)]

    for kw in ({}, {"kv": "native"}, {"neox": 0}):
        a, b = _both(monkeypatch, lambda: write(**kw))
        assert isinstance(a, list) and all(torch.equal(x, y) for x, y in zip(a, b))
    for swap in ({"positions": lambda t: t.int()}, {"key": lambda t: t[:5]}, {"key_scales": lambda t: t.half()},
                 {"query": lambda t: t.requires_grad_()}, {"value": lambda t: t.cpu()}):
        a, b = _both(monkeypatch, lambda: write(**swap))
        assert isinstance(a, tuple) and a == b


def test_calls_follow_the_current_stream():
    c = _case("native", 64)
    want = _extended(c)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)
        c.query.zero_()
        got = _extended(c)
    side.synchronize()
    assert not torch.equal(got, want)  # ordered after the side stream's zero_

"""The launches of the vector RoPE + paged K/V write, and their lanes, walked on the host.

Each launch has to read every rotary item of every token once, and the K tail
and V chunks of exactly the tokens that have a slot: V rows past cache_tokens
need not exist (loom_hip.h).
"""

from __future__ import annotations

import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


GENERAL, WAVES, TOKENS = range(3)


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("rope") / "rope_vec_items.so")
    subprocess.run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-shared", "-fPIC",
                    f"-I{os.path.join(ROOT, 'attnarc_amd', 'csrc')}",
                    os.path.join(ROOT, "tests", "rope_vec_items.cpp"), "-o", out], check=True)
    return ctypes.CDLL(out)


@pytest.mark.parametrize("cache_tokens", [0, 1, 5, 9])
@pytest.mark.parametrize("query_heads,kv_heads,rot,tail,value", [
    (32, 8, 8, 0, 16),     # 32/8 heads, head size 128, BF16
    (12, 2, 4, 0, 8),      # 72 items: a wave and eight lanes
    (1, 1, 1, 6, 8),       # 16 items, one rotary chunk a head
    (4, 4, 4, 4, 0x10),
    (3, 3, 2, 24, 32),     # long unrotated tails
    (71, 1, 5, 0, 10),     # chunk counts that no power of two divides
    (64, 64, 64, 0, 1000),  # over 2^16 items a token: plain division
])
def test_every_item_once(shim, cache_tokens, query_heads, kv_heads, rot, tail, value):
    tokens = 9
    slots = np.array([3, -1, 0, 32, 31, 7, -5, 1, 9], dtype=np.int64)  # 2 blocks of 16 tokens
    rotary = (query_heads + kv_heads) * rot
    items = rotary + kv_heads * (tail + value)
    counts = np.zeros((tokens, items), dtype=np.uint8)
    status = shim.walk_items(tokens, cache_tokens, slots.ctypes.data_as(ctypes.c_void_p), 2, 16, query_heads,
                             kv_heads, rot, tail, value, counts.ctypes.data_as(ctypes.c_void_p))
    assert status == 0
    want = np.zeros_like(counts)
    want[:, :rotary] = 1
    want[[t for t in range(cache_tokens) if 0 <= slots[t] < 32], rotary:] = 1
    np.testing.assert_array_equal(counts, want)


def _plan(shim, tokens, query_heads, kv_heads, rot, tail, value, nbytes=0, fp8=0, whole_lines=1):
    out = (ctypes.c_uint32 * 4)()
    shim.plan_of(*(ctypes.c_uint64(x) for x in (tokens, query_heads, kv_heads, rot, tail, value, nbytes, fp8,
                                                whole_lines)), out)
    return tuple(out)


@pytest.mark.parametrize("tokens,query_heads,rot,kernel", [
    (1, (1 << 31) - 2, 1, WAVES),      # 2^31 chunks a token
    (1, (1 << 31) - 1, 1, GENERAL),    # one more
    (1, (1 << 32) - 1, 1, GENERAL),    # numbers of 2^32 and more would wrap
    (1, (1 << 32) - 1, 64, GENERAL),
    (20_000_000, 62, 1, WAVES),        # 64 chunks a token
    (16_777_215, 254, 1, WAVES),       # 256 chunks: one workgroup a token, the last launch that fits
    (16_777_216, 254, 1, GENERAL),     # 2^32 threads either way
    (13_500_000, 318, 1, TOKENS),      # 320 chunks: 80 lanes' waves would be 1.3 workgroups a token
    (13_421_772, 318, 1, WAVES),
    (16_777_216, 318, 1, GENERAL),
])
def test_launch_and_index_limits(shim, tokens, query_heads, rot, kernel):
    got, _, groups, splits = _plan(shim, tokens, query_heads, 1, rot, 0, 1)
    assert got == kernel
    if got != GENERAL:
        items = (query_heads + 1) * rot + 1
        need = -(-tokens * -(-items // 64) // 4) if got == WAVES else tokens * splits
        assert groups == need and groups * 256 < 1 << 32


@pytest.mark.parametrize("heads,head_size,rotary,fp8,tokens,kernel,hint", [
    # Shapes that were slower on the other kernel, or with the hint (BF16 rows): us at each line of the rule, chosen
    # against the other.
    ((32, 32), 64, 64, 0, 10463, TOKENS, 0),    # 60 against 69 (73 with the hint)
    ((32, 32), 128, 64, 1, 8138, TOKENS, 0),    # 73 against 93 (95)
    ((16, 16), 128, 64, 0, 8000, TOKENS, 0),    # 32 against 34
    ((20, 20), 80, 80, 0, 4464, TOKENS, 0),     # 18.2 against 19.6
    ((32, 8), 128, 128, 0, 3756, TOKENS, 0),    # 18.1 against 19.0
    ((32, 8), 128, 128, 1, 4000, WAVES, 0),     # 18.8 against 19.6
    ((16, 16), 128, 128, 0, 418, WAVES, 0),     # 4.4 against 5.0
    ((32, 8), 80, 80, 0, 1802, WAVES, 0),       # 8.4 against 11.3
    ((12, 2), 64, 64, 0, 32768, WAVES, 0),      # 28 against 51
    ((32, 8), 96, 48, 0, 22977, WAVES, 0),      # 100 against 135 with the hint
    ((8, 8), 96, 48, 0, 35511, WAVES, 0),       # 87 against 124 with the hint
    ((32, 8), 128, 128, 0, 32768, WAVES, 1),    # 149 against 168
])
def test_kernel_and_hint(shim, heads, head_size, rotary, fp8, tokens, kernel, hint):
    hq, hkv = heads
    rot, tail, value = rotary // 2 // 8, (head_size - rotary) // 8, head_size // 8
    row = 2 * (hq + hkv) * rotary * 2 + hkv * (2 * head_size - rotary) * 2 + 2 * hkv * head_size * (1 if fp8 else 2)
    got = _plan(shim, tokens, hq, hkv, rot, tail, value, row * tokens, fp8, rotary * 2 % 128 == 0)
    assert got[:2] == (kernel, hint)

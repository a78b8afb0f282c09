"""The lanes of the vector RoPE + paged K/V write, walked on the host.

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


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("rope") / "rope_vec_items.so")
    subprocess.run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-shared", "-fPIC",
                    f"-I{os.path.join(ROOT, 'attnarc_amd', 'csrc')}",
                    os.path.join(ROOT, "tests", "rope_vec_items.cpp"), "-o", out], check=True)
    return ctypes.CDLL(out).walk_items


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
def test_every_item_once(walk, cache_tokens, query_heads, kv_heads, rot, tail, value):
    tokens = 9
    slots = np.array([3, -1, 0, 32, 31, 7, -5, 1, 9], dtype=np.int64)  # 2 blocks of 16 tokens
    rotary = (query_heads + kv_heads) * rot
    items = rotary + kv_heads * (tail + value)
    counts = np.zeros((tokens, items), dtype=np.uint8)
    status = walk(tokens, cache_tokens, slots.ctypes.data_as(ctypes.c_void_p), 2, 16, query_heads, kv_heads, rot, tail,
                  value, counts.ctypes.data_as(ctypes.c_void_p))
    assert status == 0
    want = np.zeros_like(counts)
    want[:, :rotary] = 1
    want[[t for t in range(cache_tokens) if 0 <= slots[t] < 32], rotary:] = 1
    np.testing.assert_array_equal(counts, want)

"""FP8 caches on the streaming kernels at the edges of their 32-token steps.

A step is two halves of 16 rows, the second one absent when the partition ends
in the first. Lengths, partitions and block sizes here end steps on every side
of a half; cache slots that hold no token are NaN codes, which no result may
see. Compared with the CPU oracle at the 16-bit bars of the other parity tests.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from attnarc_amd import ops, workloads
from gpu_util import LSE_TOL, assert_parity, oracle_expected

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EDGES = [1, 15, 16, 17, 31, 32, 33, 48, 49, 63, 65, 95, 97, 300]


def _check(lengths, heads, head_size, dtype, kernel, layout="NHD", block_size=16, partition=0):
    case = workloads.make_case(
        name="fp8", dtype=dtype, sequences=len(lengths), query_heads=heads[0], kv_heads=heads[1],
        head_size=head_size, value_head_size=head_size, block_size=block_size, lengths=lengths, seed=9, device=DEV,
        cache_encoding="fp8", layout=layout, pool_factor=1.25, partition_tokens=partition)
    expected, want_lse = oracle_expected(case)
    live = torch.zeros((case.num_blocks, block_size), dtype=torch.bool, device=DEV)
    for s, length in enumerate(lengths):
        for b in range(-(-length // block_size)):
            live[int(case.block_tables[s, b]), : length - b * block_size] = True
    dead = ~(live[:, :, None, None] if layout == "NHD" else live[:, None, :, None])
    for cache in (case.key_cache, case.value_cache):
        raw = cache.view(torch.uint8)
        raw.masked_fill_(dead.expand(raw.shape), 0x7F)
    out, lse = workloads.run_case(case, return_lse=True)
    torch.cuda.synchronize()
    assert ops.last_kernel_name() == kernel
    assert_parity(out, expected, dtype, kernel)
    np.testing.assert_allclose(lse.cpu().numpy(), want_lse, **LSE_TOL)


@pytest.mark.parametrize("head_size", [64, 80, 96, 112, 128, 256])
@pytest.mark.parametrize("layout,block_size,partition,lengths", [
    ("NHD", 16, 0, EDGES),                          # four waves per item, some without a step
    ("HND", 32, 48, EDGES),                         # partitions of one and a half steps
    ("NHD", 64, 16, [1, 16, 17, 40]),               # partitions of half a step
    ("HND", 16, 0, [1, 16, 31, 100]),               # under eight 16-token steps: one wave per item
])
def test_small_grids(head_size, layout, block_size, partition, lengths):
    _check(lengths, (6, 2), head_size, torch.float16, "decode_stream_kernel", layout, block_size, partition)


@pytest.mark.parametrize("head_size", [64, 80, 96, 112, 128])
@pytest.mark.parametrize("partition", [128, 144])
def test_grouped_workgroups(head_size, partition):
    # 1,120+ items of 8 or 9 steps of 16, ragged; head size 128 folds pairs of partitions
    _check([900, 17, 129, 513, 271, 1, 33] * 8, (8, 4), head_size, torch.bfloat16, "decode_stream_group_kernel",
           partition=partition)


@pytest.mark.parametrize("group,head_size", [(17, 64), (32, 128), (33, 128), (48, 64), (64, 128), (71, 64), (96, 128),
                                             (128, 128)])
@pytest.mark.parametrize("partition", [0, 48])
def test_wide_groups(group, head_size, partition):
    _check(EDGES, (group, 1), head_size, torch.bfloat16, "decode_stream_heads_kernel", partition=partition)

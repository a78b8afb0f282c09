"""Streaming waves with one pipeline stage, on grids large enough to take them.

At head size 128 FP8 items from 2,048 (1,024 as pairs of partitions) and at 256
FP8 items from 1,024 and 16-bit ones from 1,281 run on waves that refill their only
stage after each step. (The 16-bit rows at 128 are too short for it: they run two
stages. test_gpu_stream_plans.py has the shapes of every launch.) Ragged lengths end
items in every step remainder. Against the CPU oracle at the bars of the other
parity tests.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from attnarc_amd import ops, workloads
from gpu_util import LSE_TOL, assert_parity, oracle_expected

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("kv", ["native", "fp8"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sequences,heads,head_size,partition,kernel", [
    (255, (6, 3), 128, 128, "decode_stream_group_kernel"),  # 2,295 items, an odd head count
    (260, (16, 8), 128, 0, "decode_stream_group_kernel"),   # 2,080 whole sequences
    (516, (8, 8), 128, 512, "decode_stream_group_kernel"),  # 4,128 whole sequences
    (171, (16, 8), 128, 512, "decode_stream_group_kernel"),  # 1,368 whole sequences: two stages
    (259, (4, 2), 256, 128, "decode_stream_kernel"),        # 1,554 items
    (512, (8, 4), 256, 128, "decode_stream_group_kernel"),  # 6,144 items
])
def test_large_ragged_grids(kv, dtype, sequences, heads, head_size, partition, kernel):
    lengths = [1 + (37 * i) % 300 for i in range(sequences)]
    case = workloads.make_case(
        name="one_stage", dtype=dtype, sequences=sequences, query_heads=heads[0], kv_heads=heads[1],
        head_size=head_size, value_head_size=head_size, block_size=16, lengths=lengths, seed=23, device=DEV,
        cache_encoding=kv, layout="HND" if heads[0] == 6 else "NHD", pool_factor=1.25, partition_tokens=partition)
    out, lse = workloads.run_case(case, return_lse=True)
    torch.cuda.synchronize()
    assert ops.last_kernel_name() == kernel
    expected, want_lse = oracle_expected(case, threads=8)
    assert_parity(out, expected, dtype, f"{kv} D{head_size}")
    np.testing.assert_allclose(lse.cpu().numpy(), want_lse, **LSE_TOL)

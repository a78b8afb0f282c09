"""Wide query groups whose items are shared by several rings of K/V stages.

Small grids (up to 256 or 512 items) split an item's steps over two or four
rings and combine their states in LDS. Lengths leave rings with one step less,
or none; the grids sit on both sides of the launch rule. Against the CPU oracle
at the bars of the other parity tests.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from attnarc_amd import ops, workloads
from gpu_util import LSE_TOL, assert_parity, oracle_expected

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(lengths, group, head_size, dtype, kv, partition=0):
    case = workloads.make_case(
        name="wide", dtype=dtype, sequences=len(lengths), query_heads=group, kv_heads=1, head_size=head_size,
        value_head_size=head_size, block_size=16, lengths=lengths, seed=17, device=DEV, cache_encoding=kv,
        pool_factor=1.25, partition_tokens=partition)
    out, lse = workloads.run_case(case, return_lse=True)
    torch.cuda.synchronize()
    assert ops.last_kernel_name() == "decode_stream_heads_kernel"
    expected, want_lse = oracle_expected(case, threads=8)
    assert_parity(out, expected, dtype, f"{kv} {group}/1 D{head_size}")
    np.testing.assert_allclose(lse.cpu().numpy(), want_lse, **LSE_TOL)


@pytest.mark.parametrize("kv", ["native", "fp8"])
@pytest.mark.parametrize("group,head_size", [(17, 64), (32, 128), (33, 64), (48, 128), (49, 128), (64, 64), (65, 128),
                                             (96, 64), (100, 128), (128, 64)])
@pytest.mark.parametrize("partition", [0, 80])
def test_ring_steps(kv, group, head_size, partition):
    _check([1, 16, 17, 33, 64, 65, 97, 130, 200, 385], group, head_size, torch.float16, kv, partition)


@pytest.mark.parametrize("kv", ["native", "fp8"])
@pytest.mark.parametrize("group", [20, 40, 56])
@pytest.mark.parametrize("sequences", [256, 257, 512, 513])
def test_both_sides_of_the_grid_rule(kv, group, sequences):
    _check([1 + 7 * i % 150 for i in range(sequences)], group, 128, torch.bfloat16, kv)

"""Shapes on both sides of the streaming kernels' launch rules, against the CPU oracle.

Short items shared by four waves (two for large F32 rows), four waves on one or
two stages either side of 768 items, and FP8 pairs of partitions by group size and
cache layout.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from attnarc_amd import ops, workloads
from gpu_util import LSE_TOL, assert_parity, oracle_expected

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DTYPES = {"native": torch.bfloat16, "fp8": torch.float16, "f32": torch.float32}


def _check(kv, lengths, heads, head_size, layout="NHD", partition=0):
    dtype = DTYPES[kv]
    case = workloads.make_case(
        name="rules", dtype=dtype, sequences=len(lengths), query_heads=heads[0], kv_heads=heads[1],
        head_size=head_size, value_head_size=head_size, block_size=16, lengths=lengths, seed=29, device=DEV,
        cache_encoding="fp8" if kv == "fp8" else "native", layout=layout, pool_factor=1.25,
        partition_tokens=partition)
    out, lse = workloads.run_case(case, return_lse=True)
    torch.cuda.synchronize()
    expected, want_lse = oracle_expected(case, threads=8)
    assert_parity(out, expected, dtype, f"{kv} D{head_size} {ops.last_kernel_name()}")
    np.testing.assert_allclose(lse.cpu().numpy(), want_lse, **LSE_TOL)


@pytest.mark.parametrize("kv", ["native", "fp8", "f32"])
@pytest.mark.parametrize("head_size", [64, 80, 96, 112, 128])
@pytest.mark.parametrize("longest", [17, 33, 49, 65, 81, 127])
def test_short_contexts(kv, head_size, longest):
    for sequences in (3, 65, 129):  # 12, 260 and 516 items
        _check(kv, [1 + (29 * i) % longest for i in range(sequences - 1)] + [longest], (8, 4), head_size)


@pytest.mark.parametrize("kv", ["native", "fp8"])
@pytest.mark.parametrize("head_size", [96, 128])
@pytest.mark.parametrize("sequences", [95, 96])
def test_single_waves(kv, head_size, sequences):
    _check(kv, [1 + (53 * i) % 256 for i in range(sequences)], (8, 4), head_size, partition=128)  # 760, 768 items


@pytest.mark.parametrize("layout", ["NHD", "HND"])
@pytest.mark.parametrize("group", [1, 4, 7, 8])
def test_pairs_by_group(layout, group):
    # 1,152 items of three partitions, the second of a pair often absent
    _check("fp8", [1 + (91 * i) % 384 for i in range(95)] + [384], (4 * group, 4), 128, layout, partition=128)

"""Every launch shape of the streaming decode kernels against the CPU oracle.

Which shape a call takes is looked at on the host (test_stream_plan.py, the same
list). Lengths end items in every step remainder.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from attnarc_amd import ops, workloads
from gpu_util import LSE_TOL, assert_parity, oracle_expected
from stream_plan_shapes import SHAPES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape,plan", SHAPES)
def test_launch_shapes(shape, plan, dtype):
    kv, sequences, heads, head_size, longest, partition, layout = shape
    lengths = [1 + (37 * i) % longest for i in range(sequences - 1)] + [longest]
    case = workloads.make_case(
        name="plan", dtype=dtype, sequences=sequences, query_heads=heads[0], kv_heads=heads[1],
        head_size=head_size, value_head_size=head_size, block_size=16, lengths=lengths, seed=31, device="cuda:0",
        cache_encoding=kv, layout=layout, pool_factor=1.25, partition_tokens=partition)
    out, lse = workloads.run_case(case, return_lse=True)
    torch.cuda.synchronize()
    assert ops.last_kernel_name() == ("decode_stream_group_kernel" if plan[1] > 1 else "decode_stream_kernel")
    expected, want_lse = oracle_expected(case, threads=8)
    assert_parity(out, expected, dtype, f"{shape}")
    np.testing.assert_allclose(lse.cpu().numpy(), want_lse, **LSE_TOL)

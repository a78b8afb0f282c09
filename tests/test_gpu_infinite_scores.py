"""Steps whose scores are all -inf weigh nothing, wherever a wave meets them.

Each sequence holds one run of tokens whose scores are -inf for every head (K
rows of -inf; over an FP8 cache, which has no infinity, the least E4M3 value
under a scale that overflows): a step, a tile or a partition, at every position
a wave, a ring or a partition can start from. The other tokens are ordinary, so
the oracle's result is finite, and the bars of the other parity tests apply.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from attnarc_amd import ops, workloads
from gpu_util import LSE_TOL, assert_parity, oracle_expected

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _case(dtype, kv, heads, head_size, lengths, run, block_size=16, partition=0, layout="NHD"):
    case = workloads.make_case(
        name="inf", dtype=dtype, sequences=len(lengths), query_heads=heads[0], kv_heads=heads[1],
        head_size=head_size, value_head_size=head_size, block_size=block_size, lengths=lengths, seed=37, device=DEV,
        cache_encoding=kv, layout=layout, pool_factor=1.25, partition_tokens=partition)
    case.query.abs_()
    keys = case.key_cache.view(torch.uint8) if kv == "fp8" else case.key_cache
    if kv == "fp8":  # 0 * scale for the ordinary tokens; -448 sum(q) scale below -FLT_MAX for the others
        keys.zero_()
        case.key_scales.fill_(2e36)
    low = 0xFE if kv == "fp8" else float("-inf")
    for s, length in enumerate(lengths):
        first = s * run % length
        last = min(first + run, length)
        if last - first == length:
            last -= 1  # one ordinary token is left
        for t in range(first, last):
            block = keys[int(case.block_tables[s, t // block_size])]
            (block if layout == "NHD" else block.transpose(0, 1))[t % block_size] = low
    return case


def _check(case, kernel):
    out, lse = workloads.run_case(case, return_lse=True)
    torch.cuda.synchronize()
    assert ops.last_kernel_name() == kernel
    expected, want_lse = oracle_expected(case, threads=8)
    assert np.isfinite(expected).all() and np.isfinite(want_lse).all()
    assert_parity(out, expected, case.dtype, kernel)
    np.testing.assert_allclose(lse.cpu().numpy(), want_lse, **LSE_TOL)


KINDS = [(BF16, "native"), (F16, "native"), (BF16, "fp8"), (F32, "native")]


@pytest.mark.parametrize("dtype,kv", KINDS)
@pytest.mark.parametrize("head_size", [64, 96, 128])
@pytest.mark.parametrize("longest", [40, 110, 400])  # one wave; four waves over 4-7 steps; over 25
def test_waves_of_an_item(dtype, kv, head_size, longest):
    _check(_case(dtype, kv, (8, 4), head_size, [longest - i for i in range(9)], 32 if kv == "fp8" else 16),
           "decode_stream_kernel")


@pytest.mark.parametrize("dtype,kv", KINDS[:3])
@pytest.mark.parametrize("group", [20, 48, 64, 96, 128])
def test_rings_of_a_wide_group(dtype, kv, group):
    run = 32 if kv == "fp8" else 16
    _check(_case(dtype, kv, (group, 1), 128, [300 - i for i in range(9)], run), "decode_stream_heads_kernel")


@pytest.mark.parametrize("dtype,kv", KINDS)
@pytest.mark.parametrize("heads", [(4, 4), (32, 4)])
def test_grouped_items_and_partitions(dtype, kv, heads):
    # partitions of 128 tokens, some of them -inf throughout; FP8 folds pairs of them for eight heads a KV head
    _check(_case(dtype, kv, heads, 128, [384 - i % 7 for i in range(172)], 128, partition=128),
           "decode_stream_group_kernel")


@pytest.mark.parametrize("dtype,kv", KINDS[:3])
def test_head_size_256(dtype, kv):
    _check(_case(dtype, kv, (8, 4), 256, [200 - i for i in range(9)], 32), "decode_stream_kernel")


@pytest.mark.parametrize("dtype,kv,head_size,block_size,run,kernel", [
    (BF16, "native", 128, 8, 32, "decode_mfma_kernel"), (F16, "fp8", 128, 8, 32, "decode_mfma_kernel"),
    (F32, "native", 72, 16, 64, "decode_vector_kernel"), (F16, "native", 72, 16, 64, "decode_vector_kernel")])
def test_general_kernels(dtype, kv, head_size, block_size, run, kernel):
    _check(_case(dtype, kv, (8, 4), head_size, [400 - i for i in range(7)], run, block_size), kernel)


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("parts,partition", [(3, 16), (9, 16), (40, 16)])
def test_merge_of_infinite_partitions(dtype, parts, partition):
    # value head sizes of both merge kernels
    for head_size in (64, 80):
        _check(_case(dtype, "native", (4, 2), head_size, [partition * parts - i for i in range(5)], partition,
                     partition=partition), "decode_stream_kernel")

"""F32 queries over F32 caches on the streaming kernels, against the CPU oracle.

Head sizes 64-128 with up to 16 query heads per KV head run on F32 MFMA; the
shapes here sit at the edges of its 16-token steps, of its head tile and of
its launch rules. Both sides sum in F32 or wider, so the F32 bar of the other
parity tests (1e-5) applies.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from attnarc_amd import ops, workloads
from gpu_util import LSE_TOL, assert_parity, oracle_expected

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(lengths, heads, head_size, layout="NHD", block_size=16, partition=0, seed=3):
    return workloads.make_case(
        name="f32", dtype=torch.float32, sequences=len(lengths), query_heads=heads[0], kv_heads=heads[1],
        head_size=head_size, value_head_size=head_size, block_size=block_size, lengths=lengths, seed=seed, device=DEV,
        layout=layout, pool_factor=1.25, partition_tokens=partition)


def _check(case, kernel):
    # cache slots past a sequence's end may hold anything
    for cache in (case.key_cache, case.value_cache):
        bs = case.block_size
        for s, length in enumerate(case.lengths):
            if length % bs:
                block = cache[int(case.block_tables[s, length // bs])]
                (block if case.layout == "NHD" else block.transpose(0, 1))[length % bs :] = float("nan")
    out, lse = workloads.run_case(case, return_lse=True)
    torch.cuda.synchronize()
    assert ops.last_kernel_name() == kernel
    assert ops.last_kernel_family() == "vector"  # F32 queries, whichever kernel runs
    for cache in (case.key_cache, case.value_cache):
        cache.nan_to_num_(0.0)
    expected, want_lse = oracle_expected(case)
    assert_parity(out, expected, torch.float32, kernel)
    np.testing.assert_allclose(lse.cpu().numpy(), want_lse, **LSE_TOL)


@pytest.mark.parametrize("head_size", [64, 80, 96, 112, 128])
@pytest.mark.parametrize("layout", ["NHD", "HND"])
@pytest.mark.parametrize("heads,lengths,block_size,partition", [
    ((8, 8), [1, 15, 16, 17, 253], 16, 0),      # one live head; step remainders; four waves per item
    ((32, 2), [33, 64, 100], 32, 0),            # a full head tile; one wave per item (under 8 steps)
    ((12, 4), [1, 47, 48, 49, 200], 16, 48),    # partitions of three steps, most of them empty
    ((6, 6), [700, 129, 1] * 4, 64, 128),      # 256 < items < 1024: two waves per item above head size 64
])
def test_steps_heads_and_small_grids(head_size, layout, heads, lengths, block_size, partition):
    _check(_case(lengths, heads, head_size, layout, block_size, partition), "decode_stream_kernel")


@pytest.mark.parametrize("head_size", [64, 80, 96, 112, 128])
def test_grouped_workgroups(head_size):
    # 2,688 items of 8 steps, the last of each sequence shorter; an item count that the group does not divide
    lengths = [890, 17, 128, 513, 256, 1] * 16
    _check(_case(lengths, (4, 4), head_size, partition=128), "decode_stream_group_kernel")


@pytest.mark.parametrize("what", ["group 17", "head size 256", "block size 8", "odd stride", "odd partition"])
def test_other_shapes_stay_on_the_general_kernel(what):
    heads = (17, 1) if what == "group 17" else (8, 4)
    case = _case([70, 9, 130], heads, 256 if what == "head size 256" else 128,
                 block_size=8 if what == "block size 8" else 16, partition=40 if what == "odd partition" else 0)
    if what == "odd stride":
        store = torch.zeros(case.num_blocks * (16 * 4 * 128 + 2), device=DEV)
        view = store.as_strided(case.key_cache.shape, (16 * 4 * 128 + 2, 4 * 128, 128, 1))
        view.copy_(case.key_cache)
        case.key_cache = view
    _check(case, "decode_vector_kernel")

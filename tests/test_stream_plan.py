"""The launch shapes of streaming decode calls, on the host."""

from __future__ import annotations

import ctypes
import os
import subprocess

import pytest

from stream_plan_shapes import GROUP, GROUP_TWO, PAIRS, SHAPES, SINGLE, SINGLE_TWO, SPLIT, SPLIT_TWO

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def plan_of(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("plan") / "stream_plan.so")
    subprocess.run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-shared", "-fPIC",
                    f"-I{os.path.join(ROOT, 'attnarc_amd', 'csrc')}",
                    os.path.join(ROOT, "tests", "stream_plan.cpp"), "-o", out], check=True)
    lib = ctypes.CDLL(out)

    def plan(kv, sequences, heads, head_size, longest, partition, layout, index_order=0):
        parts = -(-longest // partition) if partition else 1
        steps = -(-(partition if parts > 1 else longest) // 16)
        got = (ctypes.c_uint32 * 4)()
        lib.plan_of(ctypes.c_uint64(sequences * parts * heads[1]), steps, head_size, heads[0] // heads[1], heads[1],
                    ctypes.c_uint64(parts), int(kv == "fp8"), int(layout == "HND"), index_order, got)
        return tuple(got)

    return plan


@pytest.mark.parametrize("shape,want", SHAPES)
def test_shapes_of_the_parity_tests(plan_of, shape, want):
    assert plan_of(*shape) == want


def test_library_split_keeps_index_order(plan_of):
    assert plan_of("native", 640, (8, 8), 128, 4096, 512, "NHD", 1) == GROUP_TWO


@pytest.mark.parametrize("shape,want", [
    # us on the shape that each took before, against this one
    (("fp8", 24, (24, 4), 128, 10202, 64, "NHD"), PAIRS),      # 56.9 on two-stage workgroups without pairs, 37
    (("fp8", 482, (32, 8), 128, 263, 64, "HND"), PAIRS),       # 134.8 on two-stage pairs, 90
    (("fp8", 401, (32, 32), 64, 17, 0, "HND"), GROUP),         # 46.1 on two stages, 39
    (("fp8", 84, (32, 32), 128, 42, 0, "HND"), SINGLE),        # 14.4 on two stages, 10.5
    (("fp8", 22, (32, 32), 128, 160, 0, "NHD"), SPLIT),        # 12.9 on two stages, 9.0
    (("fp8", 21, (20, 20), 128, 525, 512, "NHD"), SPLIT),      # 21.7 on single waves, 15.5
    (("fp8", 80, (64, 8), 112, 149, 0, "NHD"), SPLIT),         # 15.7 on two stages, 10.5
    (("native", 13, (20, 20), 96, 1310, 512, "HND"), SPLIT_TWO),  # 23.7 on single waves, 17.5
    (("native", 19, (16, 8), 80, 1325, 256, "HND"), SPLIT),    # 14.9 on single waves, 11.5
    (("native", 17, (32, 32), 256, 617, 512, "NHD"), SINGLE_TWO),  # 52.5 on one stage, 40.0
    (("native", 18, (16, 1), 128, 387, 64, "NHD"), SINGLE_TWO),  # 10.9 on four waves, 8.7
    (("native", 340, (16, 8), 128, 1000, 512, "NHD"), GROUP_TWO),  # one-stage waves up to 1.1 times as long
    (("native", 1100, (8, 8), 128, 520, 0, "HND"), GROUP_TWO),
])
def test_shapes_that_were_slower(plan_of, shape, want):
    assert plan_of(*shape) == want

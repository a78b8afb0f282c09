"""Decode shapes that take each launch shape of the streaming kernels (stream_plan.h)."""

SINGLE, SINGLE_TWO = (1, 1, 1, 0), (1, 1, 2, 0)
SPLIT, SPLIT_TWO = (4, 1, 1, 0), (4, 1, 2, 0)
GROUP, GROUP_TWO, GROUP_OF_TWO, PAIRS = (1, 4, 1, 0), (1, 4, 2, 0), (1, 2, 1, 0), (1, 4, 1, 1)

# (cache, sequences, (query heads, KV heads), head size, longest context, partition, layout) -> waves per item, items
# per workgroup, stages, pairs. Either side of each line of the rule.
SHAPES = [
    *[(("fp8", 130, (8, 4), d, 300, 0, "HND" if d == 80 else "NHD"), SPLIT) for d in (80, 96, 112, 128)],
    (("fp8", 130, (8, 4), 64, 300, 0, "NHD"), SPLIT_TWO),
    (("fp8", 128, (8, 4), 128, 300, 0, "NHD"), SPLIT_TWO),
    (("fp8", 65, (8, 4), 128, 112, 0, "NHD"), SINGLE),
    *[(("fp8", 129, (8, 4), d, 97, 0, "NHD" if d == 80 else "HND"), SINGLE) for d in (64, 80, 96, 112, 128)],
    (("fp8", 20, (16, 1), 128, 80, 0, "NHD"), SINGLE),
    (("fp8", 20, (16, 1), 128, 96, 0, "NHD"), SPLIT_TWO),
    *[(("fp8", 260, (16, 8), d, 128, 64, "HND" if d == 112 else "NHD"), GROUP) for d in (64, 80, 96, 112, 128)],
    (("fp8", 520, (8, 8), 96, 256, 0, "NHD"), GROUP),
    (("fp8", 520, (8, 8), 96, 257, 0, "NHD"), GROUP_TWO),
    (("fp8", 260, (8, 8), 96, 300, 0, "NHD"), GROUP_TWO),
    (("fp8", 180, (8, 8), 128, 150, 64, "NHD"), PAIRS),
    (("fp8", 130, (24, 4), 128, 384, 128, "NHD"), PAIRS),
    (("fp8", 130, (16, 4), 128, 384, 128, "HND"), PAIRS),
    (("fp8", 130, (16, 4), 128, 384, 128, "NHD"), GROUP_TWO),
    *[(("native", 96, (16, 8), d, 300, 0, "HND" if d == 80 else "NHD"), SPLIT) for d in (80, 96, 112, 128)],
    (("native", 96, (16, 8), 64, 300, 0, "NHD"), SPLIT_TWO),
    (("native", 191, (8, 4), 128, 300, 0, "NHD"), SPLIT_TWO),
    (("native", 96, (16, 8), 96, 400, 0, "NHD"), SPLIT_TWO),
    (("native", 96, (16, 8), 112, 400, 0, "NHD"), SPLIT),
    (("native", 20, (16, 1), 128, 96, 0, "NHD"), SINGLE_TWO),
    (("native", 20, (16, 1), 128, 112, 0, "NHD"), SPLIT_TWO),
    (("native", 20, (8, 1), 96, 64, 0, "HND"), SINGLE_TWO),
    (("native", 20, (8, 1), 96, 80, 0, "HND"), SPLIT_TWO),
    (("native", 20, (12, 2), 128, 64, 0, "NHD"), SPLIT_TWO),
    (("native", 171, (64, 16), 128, 1030, 512, "NHD"), GROUP_OF_TWO),
    (("native", 170, (64, 16), 128, 1030, 512, "HND"), GROUP_TWO),
    (("native", 320, (8, 4), 256, 200, 0, "NHD"), SINGLE_TWO),
    (("native", 321, (8, 4), 256, 200, 0, "NHD"), SINGLE),
    (("fp8", 256, (8, 4), 256, 200, 0, "NHD"), SINGLE),
]

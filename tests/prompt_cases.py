"""(rows, in_features, out_features, cherries) that the plan sends to every tile shape of the prompt-sized products, with and without a
K split: ragged rows, columns and last units; cherries within one step, over several, and over several chunks of steps.
test_prompt_plan.py holds them against the plan, test_gpu_prompt_tiles.py runs them in both widths of codes, with groups of whole
units and others: every instance of the kernels."""
SHAPE_CASES = [
    (35, 1472, 8216, 8), (33, 4128, 2784, 64), (33, 1944, 8424, 520),         # 48 x 64
    (66, 912, 11320, 112), (673, 5168, 520, 624),                             # 80 x 64
    (101, 3568, 8336, 528), (98, 5712, 4104, 56),                             # 112 x 64
    (102, 264, 8232, 8), (609, 5736, 776, 576),                               # 128 x 64
    (195, 264, 9608, 48), (85, 5768, 8232, 576),                              # 96 x 128
    (204, 264, 11856, 48), (226, 744, 11232, 528), (2023, 22392, 136, 64),    # 128 x 128
    (306, 320, 8456, 40), (289, 784, 9072, 520), (157, 6520, 8280, 8),        # 192 x 128
    (417, 272, 11016, 64), (387, 752, 11608, 544), (202, 9552, 8280, 40),     # 256 x 128
    (65, 416, 11152, 8), (681, 4520, 200, 632),                               # 48 x 64, two a compute unit
    (7, 280, 72, 8), (5, 1448, 72, 56), (5, 1720, 72, 520),                   # 16 x 64
    (5, 264, 656, 8), (5, 2264, 2144, 48), (5, 744, 544, 536),                # 16 x 64, two a compute unit
    (20, 272, 104, 8), (18, 1472, 72, 104), (19, 960, 72, 616),               # 32 x 64, shared K
    (36, 264, 8304, 8), (673, 4976, 200, 80), (51, 3504, 4104, 536),          # 64 x 64, shared K
    # 96 columns: 96 rows, 128 rows
    (306, 264, 5576, 8), (423, 344, 4176, 0), (264, 1104, 5968, 528), (85, 6824, 5616, 8), (83, 7560, 5800, 616),
    (690, 1088, 3152, 528), (193, 10168, 2880, 8), (592, 8216, 1112, 520),
    # and what of the others the plan no longer sends above
    (41, 5952, 8888, 40), (141, 1584, 7240, 8), (67, 6408, 2736, 8), (546, 5288, 2392, 232), (99, 12264, 2936, 8), (328, 976, 8736, 8),
    (98, 8976, 8248, 8), (5, 280, 4688, 8), (58, 288, 9312, 8),
]
# more tiles of 192 or 256 rows than there are compute units, so that a workgroup goes on to further ones: one unit of 128 positions, an even and an
# odd number of them, a ragged last one; no cherries, some, several chunks of steps
ROUND_CASES = [(2000, 128, 8200, 0), (2000, 264, 8200, 8), (1990, 392, 8264, 8), (1700, 1000, 12296, 40), (1500, 904, 13000, 520)]
# the same with K split: a workgroup goes on from one split's tile to another's, so that its units, cherry steps (the last split's only: none, one, two
# chunks and more) and tickets change; ragged last splits
SPLIT_ROUND_CASES = [(950, 9808, 4136, 0), (516, 11128, 7048, 136), (306, 25216, 5520, 520), (207, 23344, 12640, 40), (398, 16944, 9088, 264),
                     (395, 16424, 8304, 520)]

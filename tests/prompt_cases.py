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
]

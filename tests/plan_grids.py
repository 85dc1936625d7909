"""Grids of the tests by the form that the plan gives them (test_plans.py checks
that it does): the step's (reconstruction, tile rows, runs) and the rows of the
gather's tiles.  The FP16 modes share FP32's tiles."""

_fp32 = {
    ("tri", 12, False): [(41, 21, 44), (96, 84, 40), (150, 97, 83)],   # overlaps in x and y, in x; large
    ("tri", 12, True): [(102, 61, 41), (38, 54, 126)],
    ("tri", 8, False): [(64, 64, 32), (64, 20, 37)],
    ("tri", 4, False): [(20, 20, 20), (33, 25, 4)],
    # gradient reconstruction: grids of one plane (their own form) among them
    ("grad", 12, False): [(41, 21, 44), (96, 84, 40), (256, 300, 1)],
    ("grad", 8, False): [(64, 64, 32), (512, 96, 1)],
    ("grad", 4, False): [(20, 20, 20), (33, 25, 4), (64, 32, 1), (200, 97, 1)],
}
_fp64 = {
    ("tri", 12, False): [(48, 40, 20), (90, 50, 121)],
    ("tri", 12, True): [(82, 39, 41), (51, 50, 49)],
    ("tri", 8, False): [(64, 64, 32), (64, 20, 37)],
    ("tri", 4, False): [(20, 20, 20), (8, 64, 8)],
    ("grad", 12, False): [(48, 40, 20), (96, 84, 40), (256, 300, 1)],
    ("grad", 8, False): [(64, 64, 32), (300, 97, 1)],
    ("grad", 4, False): [(20, 20, 20), (64, 32, 1)],
}
STEP_GRIDS = {form: {"fp64": _fp64[form], "fp32": _fp32[form], "fp16": _fp32[form], "fp16n": _fp32[form]}
              for form in _fp32}

# 12 rows: 96 rows of cells leave no overlap, the other grids do; grids of one
# plane, and in FP64 of two in one chunk (forms of their own), among them
GATHER_GRIDS = {
    12: {"fp64": [(32, 40, 26), (64, 80, 64), (96, 96, 30), (512, 200, 1), (512, 200, 2), (256, 192, 2)],
         "fp32": [(32, 32, 65), (64, 80, 64), (128, 40, 128), (96, 96, 64), (512, 400, 1)],
         "fp16": [(32, 32, 65), (96, 96, 64), (512, 400, 1)]},
    8: {"fp64": [(64, 64, 32), (32, 8, 1), (96, 40, 1), (256, 200, 2)], "fp32": [(64, 64, 32), (32, 8, 1), (96, 40, 1)],
        "fp16": [(64, 64, 32), (32, 8, 1), (96, 40, 1)]},
}

"""Batches for the tests of decode attention's deal: every way to cut a batch, in each variant of
the kernel."""

# head size, query heads a kv head, fp8 cache
VARIANTS = [(64, 4, False), (128, 3, False), (128, 6, True), (256, 2, False), (256, 2, True)]

_ragged = [0 if i % 7 == 5 else 600 + i if i % 7 == 1 else (i * 37) % 150 for i in range(300)]
_ragged[3], _ragged[4], _ragged[150], _ragged[299] = 3000, 1500, 2100, 2999
_spread = [0 if i % 9 < 2 else 137 + (i * 463) % 964 for i in range(200)]

# what a variant each does on 256 CUs: least pieces (L), whole pairs (W), larger pieces (P), equal
# ranges (R); lengths, kv heads, block size, window, cap
BATCHES = [
    ("LLLLL", [3000, 17, 1, 0, 700], 2, 16, 0, 0.0),
    ("WWWWW", [700 + i for i in range(60)], 8, 16, 0, 0.0),
    ("LWLWW", [0 if i % 9 == 5 else (i * 53) % 400 for i in range(200)], 8, 32, 0, 30.0),
    ("PPPPP", [2800, 0] + [2500 + 40 * i for i in range(15)], 8, 16, 0, 0.0),
    ("PPPPP", [2800, 0] + [2500 + 40 * i for i in range(15)], 8, 32, 2400, 30.0),
    ("RRRRR", _ragged, 8, 16, 0, 0.0),
    ("RWRRR", _ragged, 3, 32, 1000, 30.0),
    ("WRWRR", _spread, 8, 16, 0, 30.0),
]

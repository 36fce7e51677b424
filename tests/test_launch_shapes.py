"""What the dispatch launches, call by call, without a GPU (tests/launches.py)."""
import re

import pytest

from launches import record, t

ROWS = [1, 8, 64, 65, 250, 256, 257, 640, 1023, 1024, 2047, 2048, 2049, 4096, 4097, 16384, 40000]
WIDTHS = [1, 3, 63, 64, 65, 100, 127, 128, 129, 192, 200, 255, 256, 257, 301, 320, 321, 384, 500, 511, 512, 513, 700, 767,
          1000, 1021, 1023, 1024, 1025, 1100, 1500, 2000, 2047, 2048, 2049, 4095, 4096, 4097, 8191, 8193, 16383, 16384,
          16385, 20000]


def test_the_causal_softmax_takes_the_form_of_the_softmax_alone():
    """The order in which a row's exps are added, and so the last bit of a
    probability, depends on the form: shp_soft_max_causal is bit for bit
    diag_mask_inf then soft_max_ext only if both take the same one."""
    calls = []
    for rows in ROWS:
        for n in WIDTHS:
            x, y = t(n, rows), t(n, rows)
            calls += [("shp_soft_max_ext", x, None, 0.5, 0.0, y), ("shp_soft_max_causal", x, 0, 0.5, y),
                      ("shp_soft_max_ext", x, t(n, rows), 0.5, 0.0, y)]
    got = record(calls)
    # k_soft_max_wave<K, MK>, k_soft_max_rows4<WPR, K4, MK, ODD, BLOCK>, k_soft_max_block<MK>
    mask = {"wave": 1, "rows4": 2, "block": 0}
    for i in range(0, len(got), 3):
        forms = []
        for st, launches in got[i:i + 3]:
            assert st == 0 and len(launches) == 1
            name, grid, block, _ = launches[0]
            kind, args = re.search(r"k_soft_max_(wave|rows4|block)I((?:L[ib]\d+E)+)E", name).groups()
            args = re.findall(r"L[ib](\d+)E", args)
            del args[mask[kind]]
            forms.append((kind, args, grid, block))
        assert forms[0] == forms[1] == forms[2], calls[i]


def _kernels(calls):
    got = record(calls)
    assert all(st == 0 for st, _ in got)
    return [[n for n, *_ in ls] for _, ls in got]


def test_short_odd_softmax_rows_go_by_elements_while_they_are_few():
    sizes = [(16, 129), (1024, 201), (4096, 319), (2048, 321), (1, 511), (4097, 319), (2049, 321), (2049, 511), (16, 513),
             (16, 300), (100000, 129)]
    names = _kernels([("shp_soft_max_ext", t(n, rows), None, 0.5, 0.0, t(n, rows)) for rows, n in sizes])
    assert ["k_soft_max_wave" in k[0] for k in names] == [True] * 5 + [False] * 6

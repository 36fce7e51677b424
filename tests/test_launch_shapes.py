"""What the dispatch launches, call by call, without a GPU (tests/launches.py)."""
import re

import pytest

from launches import layer, record, t

ROWS = [1, 8, 64, 65, 250, 256, 257, 640, 1023, 1024, 2047, 2048, 2049, 2689, 3329, 4096, 4097, 6144, 6145, 16384, 40000]
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
            calls += [("shp_soft_max_ext", x, None, 0.5, 0.0, y), ("shp_soft_max_causal", x, 0, 0.5, y)]
    got = record(calls)
    # k_soft_max_wave<K, MK>, k_soft_max_rows4<WPR, K4, MK, ODD, BLOCK>, k_soft_max_block<MK>
    mask = {"wave": 1, "rows4": 2, "block": 0}
    for i in range(0, len(got), 2):
        forms = []
        for st, launches in got[i:i + 2]:
            assert st == 0 and len(launches) == 1
            name, grid, block, _ = launches[0]
            kind, args = re.search(r"k_soft_max_(wave|rows4|block)I((?:L[ib]\d+E)+)E", name).groups()
            args = re.findall(r"L[ib](\d+)E", args)
            del args[mask[kind]]
            forms.append((kind, args, grid, block))
        assert forms[0] == forms[1], calls[i]


def test_many_long_softmax_rows_take_one_wave_where_two_begin_another_round():
    """k_soft_max_rows4<waves, ...> of 1025 to 2048 scores, each side of every line."""
    def waves(rows, n, mask):
        x = t(n, rows)
        return ("shp_soft_max_ext", x, t(n, rows) if mask else None, 0.5, 0.0, x)
    cases = [(2688, 1601, False, 2), (2689, 1601, False, 1), (2689, 1600, False, 2), (4608, 1600, False, 2), (4609, 1025, False, 1),
             (6144, 2048, False, 1), (6145, 2048, False, 2), (4609, 1600, True, 2),
             (2688, 2048, True, 2), (2689, 1601, True, 1), (3328, 2048, True, 1), (3329, 2048, True, 2), (40000, 1025, False, 2)]
    names = _kernels([waves(*c[:3]) for c in cases])
    assert [int(re.search(r"rows4ILi(\d+)E", k[0]).group(1)) for k in names] == [c[3] for c in cases]


def _kernels(calls):
    got = record(calls)
    assert all(st == 0 for st, _ in got)
    return [[n for n, *_ in ls] for _, ls in got]


def test_short_odd_softmax_rows_go_by_elements_while_they_are_few():
    sizes = [(16, 129), (1024, 201), (4096, 319), (2048, 321), (1, 511), (4097, 319), (2049, 321), (2049, 511), (16, 513),
             (16, 300), (100000, 129)]
    names = _kernels([("shp_soft_max_ext", t(n, rows), None, 0.5, 0.0, t(n, rows)) for rows, n in sizes])
    assert ["k_soft_max_wave" in k[0] for k in names] == [True] * 5 + [False] * 6


def test_narrow_rows_take_blocks_of_their_own_width():
    """Strided rows, a value per row added and a row repeated: rows of up to a
    wave's or two waves' float4 do not launch four waves each; few short rows go
    by elements; a row is split over blocks only where the rows are few or long."""
    #       rows, width, threads, blocks per row
    shapes = [(100000, 1, 64, 1), (100000, 64, 64, 1), (100000, 65, 64, 1), (100000, 259, 64, 1), (100000, 260, 128, 1),
              (100000, 515, 128, 1), (100000, 516, 256, 1), (1024, 65, 256, 1), (512, 512, 256, 1), (513, 512, 128, 1),
              (1024, 513, 128, 1), (7, 64, 64, 1), (96, 24001, 256, 24), (2000, 12001, 256, 12), (20000, 12001, 256, 1),
              (2000, 2000, 256, 1)]
    def calls(rows, n):
        x, y, pad = t(n, rows, nb=[4, 4 * n + 12]), t(n, rows), t(n, rows, nb=[4, 4 * n + 4])
        return [("shp_sqr", x, pad), ("shp_add", y, t(n), pad), ("shp_add", x, t(1, rows), y),
                ("shp_glu_swiglu", t(2 * n, rows), 0, y)]
    got = record([c for rows, n, *_ in shapes for c in calls(rows, n)])
    for i, (rows, n, block, runs) in enumerate(shapes):
        for st, ls in got[4 * i:4 * i + 4]:
            assert st == 0 and len(ls) == 1 and "_rows" in ls[0][0]
            assert (ls[0][2], ls[0][1]) == ((block, 1, 1), (min(rows, 65536), runs, 1)), (rows, n, ls)


def test_short_row_sums_and_norms_go_by_elements():
    """Up to 128 elements a row sum, up to 64 a norm: no float4 (the last template
    argument), whatever their count; a row of up to 1024 is one wave's batch of loads."""
    def last(name):
        return int(re.findall(r"Li(\d+)E", name)[-1])
    for rows in (1, 300, 2048, 100000):
        for op, widths in (("shp_sum_rows", {1: 0, 7: 0, 64: 0, 127: 0, 128: 0, 129: 1, 259: 1, 260: 2, 515: 2, 516: 4, 1027: 4}),
                           ("shp_norm", {1: 0, 6: 0, 63: 0, 64: 0, 65: 1, 259: 1})):
            extra = (1e-5,) if op == "shp_norm" else ()
            names = _kernels([(op, t(n, rows), *extra, t(n if extra else 1, rows)) for n in widths])
            assert [last(k[0]) for k in names] == list(widths.values()), (op, rows, names)
            assert op == "shp_norm" or all("Li64E" in k[0] for k in names)


def _istft(n, hop, frames):
    return "shp_inverse_stft", t(n + 2, frames), n, hop, t((frames - 1) * hop)


def test_inverse_stft_forms_its_frames_once_only_where_the_blocks_are_long_enough():
    """Windows whose LDS leaves a block few samples go sample by sample once the
    chip is full; blocks get longer with the utterance."""
    cases = [((400, 100, 20), False), ((400, 100, 4801), True), ((512, 204, 2400), True), ((200, 25, 80000), True),
             ((360, 72, 6000), True), ((540, 216, 9000), True), ((600, 600, 800), True), ((20, 5, 24001), False),
             ((256, 64, 2000), False), ((512, 512, 29), False)]
    names = _kernels([_istft(*c) for c, _ in cases])
    assert [("k_istft_direct" in k[0]) for k in names] == [d for _, d in cases]
    per_block = []
    for frames in (300, 6000, 24001, 400000):
        (st, ls), = record([_istft(20, 5, frames)])
        per_block.append(-(-(frames - 1) * 5 // ls[0][1][0]))
    assert per_block == sorted(per_block) and per_block[0] <= 64 and per_block[-1] > 400, per_block


def test_log_mel_spreads_its_frames_over_the_chip():
    """Few frames go a block each (a short transform in the block-per-frame form),
    more in as few blocks as one a CU."""
    def call(n, hop, frames, bins=80):
        ns = (frames - 1) * hop + n - 2 * ((n - hop) // 2)
        return "shp_log_mel", t(ns), t(n // 2 + 1, bins), n, hop, n, t(bins, frames)
    #        n_fft, hop, frames, frame form, blocks
    cases = [(64, 16, 250, True, 250), (64, 16, 1536, True, 1536), (64, 16, 1537, False, 193), (256, 64, 384, True, 384),
             (256, 64, 385, False, 193), (16, 4, 2049, False, 129), (1024, 256, 15, False, 15), (1024, 256, 256, False, 256),
             (1024, 256, 257, False, 129), (1024, 256, 937, False, 235), (1024, 256, 2000, False, 500), (2048, 512, 900, False, 900),
             (1, 1, 100, False, 100), (512, 128, 1875, False, 235)]
    got = record([call(*c[:3]) for c in cases])
    for (n, hop, frames, form, blocks), (st, ls) in zip(cases, got):
        assert st == 0 and len(ls) == 1
        assert (("k_log_mel_frame" in ls[0][0]), ls[0][1][0]) == (form, blocks), (n, frames, ls)
        assert ls[0][3] <= 64 * 1024


def _layer_step(T, hidden=4, heads=1, kv=1, ffn=4):
    x = lambda n: t(n, T)
    w = lambda n: t(n, type_=30)
    q, k = lambda: t(128, heads, T), lambda: t(128, kv, T)
    return "shp_layer_nongemm_step", layer(x(hidden), w(hidden), x(hidden), q(), k(), w(128), w(128), t(T, type_=26), q(), k(),
                                           x(hidden), w(hidden), x(hidden), x(hidden), x(ffn), x(ffn), x(ffn), x(hidden), x(hidden))


def test_a_launch_ends_below_two_to_the_32_threads():
    """Tensors of more rows, samples or positions than one launch's threads: several
    launches that together have a block for all of it (the step: its five). Those
    of 2^26 rows and more ended in an error before any split."""
    def soft(n, rows, causal):
        x, y = t(n, rows), t(n, rows)
        return ("shp_soft_max_causal", x, 0, 0.5, y) if causal else ("shp_soft_max_ext", x, None, 0.5, 0.0, y)
    #        call, blocks in all
    cases = [(("shp_norm", t(300, 50000001), 1e-5, t(300, 50000001)), 25000001),
             (("shp_norm", t(700, 20000000), 1e-5, t(700, 20000000)), 5000000),
             (("shp_norm", t(70000, 5000001), 1e-5, t(70000, 5000001)), 5000001),
             (soft(9001, 5000003, False), 5000003), (soft(9001, 5000003, True), 5000003),
             (soft(2047, 60000001, False), 30000001), (soft(17000, 4500000, False), 4500000), (soft(130, 80000001, False), 20000001),
             (("shp_log_mel", t(9000000), t(1025, 8), 2048, 1, 2048, t(8, 8999999)), 8999999),
             (_istft(160, 20, 100000001), None), (_istft(20, 5, 400000001), None), (_istft(400, 100, 20000001), None)]
    for (call, blocks), (st, ls) in zip(cases, record([c for c, _ in cases])):
        assert st == 0 and ls, (call[0], st)
        for _, grid, block, _ in ls:
            assert grid[0] * block[0] < 2 ** 32 and grid[1:] == block[1:] == (1, 1), (call, ls)
        assert blocks is None or sum(g[0] for _, g, *_ in ls) == blocks, (call, ls)
        assert len({n for n, *_ in ls}) == 1 and len(ls) == -(-sum(g[0] for _, g, *_ in ls) // ((2 ** 32 - 1) // ls[0][2][0]))
    for T in (100, 8388607, 8388608, 9000000):
        (st, ls), = record([_layer_step(T)])
        assert st == 0 and all(g[0] * b[0] < 2 ** 32 for _, g, b, _ in ls)
        assert len(ls) == (1 if T <= 8380000 else 5), (T, ls)


def test_im2col_reads_a_window_by_value_only_where_that_is_ahead():
    """The window walk (the last template argument: 0 by value, 1 four samples, 2 four
    channels) by layout, and for F16 columns by bank conflicts, taps and size."""
    def walk(x, k, d, ow, type_=0, s0=1):
        c = x["ne"][1]
        (st, ls), = record([("shp_im2col", t(k, c), x, s0, 0, d, t(c * k, ow, type_=type_))])
        assert st == 0
        return int(re.findall(r"Li(\d+)E", ls[0][0])[-1])
    for L, C, k, d, s0, f16, want in [(4136, 256, 3, 1, 1, 0, 1), (65536, 64, 3, 1, 1, 0, 1), (4097, 256, 3, 1, 1, 1, 1), (4098, 256, 3, 1, 1, 1, 0),
                                      (65536, 127, 3, 1, 1, 1, 0), (65536, 128, 3, 1, 1, 1, 1), (4136, 256, 4, 1, 1, 1, 0), (4136, 256, 5, 1, 1, 1, 1),
                                      (65536, 64, 16, 1, 4, 1, 0), (65536, 47, 1, 1, 1, 1, 1), (65536, 48, 1, 1, 1, 1, 0), (65536, 64, 11, 1, 1, 1, 1), (500, 64, 3, 5, 1, 1, 0), (500, 64, 3, 3, 1, 1, 0),
                                      (500, 64, 3, 2, 1, 1, 1), (500, 64, 3, 5, 1, 0, 1), (500, 31, 3, 5, 1, 1, 1), (500, 32, 3, 5, 1, 1, 0),
                                      (250000, 31, 3, 1, 1, 1, 1),
                                      (24000, 1, 16, 1, 8, 1, 1)]:
        assert walk(t(L, C), k, d, (L - (k - 1) * d - 1) // s0 + 1, f16, s0) == want, (L, C, k, d, s0, f16)
    for f16 in (0, 1):
        assert walk(t(1000, 80, nb=[4 * 80, 4]), 3, 1, 998, f16) == 2       # channel-major
        assert walk(t(1000, 80, nb=[8, 8000]), 3, 1, 998, f16) == 0         # every other sample

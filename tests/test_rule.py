"""The granularity rule (x-ted_amd/csrc/device.hpp) on the host: which class a
table of given sides, nesting and leaves takes, and what a caller's settings
promise about it."""
import ctypes
import inspect
import itertools
import os
import random
import subprocess

import numpy as np
import pytest

import autotune
import xted
from conftest import ROOT

NO_FORM, FIRST_XL, LDS_MAX = 26, 27, 150 * 1024


class Rule(ctypes.Structure):
    _fields_ = [(f, ctypes.c_int) for f in
                ("lds_per_wave", "max_cpl", "min_waves", "wide_cols", "tail")]


class Table(ctypes.Structure):
    _fields_ = [(f, ctypes.c_int) for f in ("a", "b", "kd_r", "kd_c", "leaves_c")] + \
               [("cells", ctypes.c_longlong)]


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("rule") / "rule.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC",
                    os.path.join(ROOT, "tests", "rule_shim.cpp"), "-o", so], check=True)
    return ctypes.CDLL(so)


def classify(shim, table, rule=None, force=-1):
    """(class, LDS bytes) of Table fields under Rule fields (the default's)."""
    need = ctypes.c_longlong()
    r = Rule(*(rule or (10 * 1024, 16, 1, 1 << 30, 0)))
    cls = shim.rule_class(ctypes.byref(r), ctypes.byref(Table(*table)), force, ctypes.byref(need))
    return cls, need.value


def tables(seed, count):
    """Tables of every size a rule tells apart, short and tall, shallow and
    deep, in levels of few and of many cells."""
    rnd = random.Random(seed)
    sides = [2, 3, 16, 17, 33, 64, 65, 128, 256, 257, 400, 512, 513, 1000, 1024, 1025, 2000, 2048,
             2049, 3000, 4096, 4097, 8000, 8192, 8193, 12000, 20000]
    for _ in range(count):
        a, b = rnd.choice(sides), rnd.choice(sides)
        rows, cols = min(a, b), max(a, b)
        kd_r = min(rnd.choice([1, 2, 5, 20, 60]), (rows - 1) // 2)
        kd_c = min(rnd.choice([1, 2, 5, 20, 60, 120, 250, 550]), (cols - 1) // 2)
        leaves = max(kd_c + 1, min(cols - kd_c, rnd.choice([2, 10, cols // 4, cols // 2, cols - 1])))
        yield a, b, kd_r, kd_c, leaves, rows * cols * rnd.choice([1, 10, 500, 5000])


def test_forced_row_class_takes_every_table_that_fits(shim):
    """Whatever the rule would choose: column blocks for tall tables, one
    wave's sweep for short ones of a large level. (A table takes shared slot
    rows only where no row-scan class fits it.)"""
    replaced = set()
    for t in tables(1, 6000):
        cols = max(t[0], t[1])
        auto, _ = classify(shim, t)
        for waves, cpl in itertools.product((1, 2, 4, 8, 16), (1, 2, 4, 8, 16)):
            cls = 1 + 5 * (waves.bit_length() - 1) + (cpl.bit_length() - 1)
            need = shim.scan_need(max(t[2], 1), t[4], t[3], waves)
            fits = cols <= min(64 * waves * cpl, 8192) and need <= LDS_MAX
            got, lds = classify(shim, t, force=cls)
            if auto != NO_FORM and fits:
                assert (got, lds) == (cls, need), (t, waves, cpl)
                replaced.add(auto)
            else:
                assert got == auto
    assert replaced & set(range(FIRST_XL, FIRST_XL + 6)) and xted.CLASS_SWEEP in replaced
    assert not replaced & {xted.CLASS_SHARED + k for k in range(3)}


def test_forced_blocks_and_tiny_forms(shim):
    for t in tables(2, 3000):
        auto, _ = classify(shim, t)
        for force in list(range(FIRST_XL, FIRST_XL + 6)) + [xted.CLASS_TINY + k for k in range(3)]:
            got, lds = classify(shim, t, force=force)
            assert got == force or got == auto
            if got == force and force >= xted.CLASS_TINY:
                k = force - xted.CLASS_TINY
                assert max(t[0], t[1]) <= xted.TINY_SEG[k] and lds <= 2048 << k
            if auto == NO_FORM:
                assert got == NO_FORM


def waves_and_columns(cls, cols):
    """Waves of a table of class cls and the columns a lane of them holds."""
    if 1 <= cls <= 25:
        waves, cpl = 1 << (cls - 1) // 5, 1 << (cls - 1) % 5
        return waves, cpl
    if xted.CLASS_SHARED <= cls < xted.CLASS_SWEEP:
        return 4 << (cls - xted.CLASS_SHARED), 8
    if FIRST_XL <= cls < FIRST_XL + 6:
        k = cls - FIRST_XL
        blocks = -(-cols // xted.XL_BW[k])
        return (8, 8, 8, 4, 1, 1)[k] * blocks, (8, 4, 2, 2, 4, 2)[k]
    return 1, 1


@pytest.mark.parametrize("max_cpl", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("min_waves,wide_cols", [(1, 1 << 30), (2, 600), (3, 300), (16, 1025)])
def test_settings_hold_for_every_class(shim, max_cpl, min_waves, wide_cols):
    """Tables of at least wide_cols columns get at least min_waves waves, and
    every table as many as max_cpl columns a lane take (16 at most)."""
    seen = set()
    for t in tables(3, 6000):
        cols = max(t[0], t[1])
        cls, _ = classify(shim, t, (10 * 1024, max_cpl, min_waves, wide_cols, 0))
        seen.add(cls)
        if cls == NO_FORM or xted.CLASS_TINY <= cls < xted.CLASS_SHARED:
            continue
        on_chip = cls <= 25 or cls >= xted.CLASS_SHARED
        waves, _ = waves_and_columns(cls, cols)
        # (Column blocks are also where tables go that fit nothing else.)
        if cols >= wide_cols and (on_chip or cls == FIRST_XL + 2):
            assert waves >= min_waves, (t, cls)
        if cls != xted.CLASS_SWEEP and on_chip:
            assert waves >= min(16, -(-cols // (64 * max_cpl))), (t, cls)
        if cls == xted.CLASS_SWEEP:
            assert max_cpl >= 8
    assert {xted.CLASS_SHARED + k for k in range(3)} & seen
    assert max_cpl < 8 or min_waves > 1 or xted.CLASS_SWEEP in seen


def test_deep_tables_of_one_workgroup_stay_in_it(shim):
    """Blocks of one wave take no table of up to 2048 columns that one
    workgroup holds: their rows wait for each other longer than they save."""
    one_wave = {FIRST_XL + 4, FIRST_XL + 5}
    taken = {xted.CLASS_SHARED: 0, "on chip": 0}
    for t in itertools.product((300, 500, 900), (350, 500, 1000, 1500, 2000, 2048), (20, 60, 100),
                               (100, 150, 200, 250), (300, 450), (1 << 18, 1 << 22)):
        if t[3] >= min(t[4], t[1] // 2) or t[4] > t[1] or t[0] > t[1] or t[2] >= t[0] // 2:
            continue
        if shim.scan_need(t[2], t[4], t[3], 1) > LDS_MAX:
            continue
        cls, _ = classify(shim, t, (10 * 1024, 16, 1, 1 << 30, 1))
        assert cls not in one_wave, t
        taken[xted.CLASS_SHARED] += cls == xted.CLASS_SHARED
        taken["on chip"] += cls <= 25
    assert all(taken.values())


def test_every_table_that_fits_lds_has_a_form(shim):
    """Under any settings: a table of up to 8192 columns whose slot rows fit
    one workgroup is taken."""
    for max_cpl, min_waves in ((16, 1), (8, 1), (8, 16), (16, 7)):
        for t in tables(4, 6000):
            if max(t[0], t[1]) <= 8192 and shim.scan_need(max(t[2], 1), t[4], t[3], 1) <= LDS_MAX:
                for tail in (0, 1):
                    cls, need = classify(shim, t, (10 * 1024, max_cpl, min_waves, 600, tail))
                    assert cls != NO_FORM and need <= LDS_MAX + 10 * 1024, t


def test_python_defaults_are_a_new_contexts(shim):
    """Context.set_tuning() restores a new context's rule, and the tuner's
    baseline (also what load() gives without a stored rule) is that rule."""
    out = (ctypes.c_int * 9)()
    shim.default_knobs(out)
    keys = ["lds_per_wave", "max_cpl", "min_waves", "wide_cols", "tail_pairs", "level_align",
            "size_bands", "light_lds", "tiny_forms"]
    knobs = dict(zip(keys, out))
    assert autotune.DEFAULT == knobs
    assert autotune.load("/nonexistent/tuning.json") == knobs
    for method, names in (("set_tuning", keys[:4]), ("set_size_bands", ["size_bands"]),
                          ("set_tiny_forms", ["tiny_forms"])):
        params = list(inspect.signature(getattr(xted.Context, method)).parameters.values())[1:]
        assert [p.default for p in params] == [knobs[k] for k in names], method


def test_tuner_starts_from_the_default(monkeypatch, tmp_path):
    """The command's search has a new context's rule to beat."""
    started = []

    def fake_tune(ctx, xs, ys, **kw):
        started.append(kw["start"])
        return dict(kw["start"]), [], 0.0

    class FakeContext:
        def __init__(self, device):
            pass

        def __enter__(self):
            return self

        def __exit__(self, *exc):
            pass

        def pool_add(self, trees):
            return np.arange(len(trees))

    monkeypatch.setattr(autotune, "tune", fake_tune)
    monkeypatch.setattr(autotune.xted, "Context", FakeContext)
    monkeypatch.setattr("sys.argv", ["autotune", "--pairs", "2", "--out", str(tmp_path / "t.json")])
    autotune.main()
    assert started == [autotune.DEFAULT]
    assert autotune.load(str(tmp_path / "t.json")) == autotune.DEFAULT

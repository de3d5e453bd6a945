"""The launch rules on the host: what a launch chooses fits the GPU it is for.  No GPU needed."""
import pytest

import launchtools as L

LDS = 160 * 1024  # bytes a workgroup may use on gfx950


@pytest.fixture(scope="module")
def metadata():
    pytest.importorskip("msgpack")
    return L.kernel_metadata()


@pytest.mark.parametrize("batched", [0, 1])
@pytest.mark.parametrize("strategy", ["exact", "fast", "half"])
@pytest.mark.parametrize("radius", [1.2, 1.9])
def test_table_and_state_fit_lds(metadata, batched, strategy, radius):
    """Tables around every kernel's limit: the chosen kernel's own LDS and the table's together
    stay within the 160 KiB of a workgroup."""
    tables = [100, 10238, 10239, 10240, *range(10740, 10756), 11774, 11775, 11776, 11777]
    kernels = [0, L.PAIR, L.CARRY, L.STAGED]
    cases = [{"box": 128, "spaces": 50, "radius": radius, strategy: 1, "batched": batched,
              "table": n, "kernel": k} for n in tables for k in kernels
             if not (batched and n > 11776)]
    for case, (which, _, _, lds, symbol) in zip(cases, L.choices(cases)):
        assert symbol in metadata, case
        assert metadata[symbol][".group_segment_fixed_size"] + lds <= LDS, (case, which, symbol)


def test_largest_table_of_the_carried_queues():
    """The carried queues take tables up to what 160 KiB leave beside their state; a batch's launch
    keeps a count there too, so its limit is a few samples lower."""
    cases = [{"box": 128, "spaces": 50, "fast": 1, "batched": b, "table": n, "kernel": L.CARRY}
             for b in (0, 1) for n in (10747, 10748, 10751, 10752)]
    got = [c[0] for c in L.choices(cases)]
    assert got == [L.CARRY, L.CARRY, L.CARRY, L.PAIR, L.CARRY, L.PAIR, L.PAIR, L.PAIR]


@pytest.mark.parametrize("case,first", [({"fast": 1}, "2,0"), ({"fast": 1, "bounded": 1}, "1,0"),
                                        ({"half": 1}, "1,0"), ({"half": 1, "bounded": 1}, "1,0")])
def test_batch_tuner_times_each_kernel_and_box_once(case, first):
    """Fast math: the schedules run by the kernel such launches run by default, by its name; over the
    fastest, per-pair and carried kernel with sliding and fixed boxes, each combination once."""
    *got, schedules = L.ask("batch_tuner", [case])[0]
    assert got[0] == first and sorted(got) == ["1,0", "1,1", "2,0", "2,1"]
    assert int(schedules) == 24


def test_batch_tuner_exact():
    got = L.ask("batch_tuner", [{}])[0]
    assert got == ["0,0", "6"]  # the schedules; one kernel


def test_op_tuner_times_schedules_where_the_default_is_cells():
    """Where the default kernel may be the small-problem kernel, which runs no schedule, every
    schedule names a brick kernel; elsewhere fast math leaves the kernel to the launch."""
    fast, half, exact, plain = L.ask("op_tuner", [{"fast": 1, "cells": 1}, {"half": 1, "cells": 1},
                                                  {"cells": 1}, {"fast": 1}])
    assert set(fast) == {str(L.CARRY)} and set(half) == {str(L.PAIR)} and set(plain) == {"0"}
    assert set(exact) == {str(L.STAGED), str(L.PAIR)}
    assert len(fast) == len(half) == len(exact) == len(plain) == 24


def test_tuning_keys_name_all_that_a_launch_depends_on():
    """Lines written when a knob meant another launch have other keys; so have launches whose depth
    scale or cells differ by what Init was told, and bounded and unbounded batches."""
    old_op, old_batch = "k2:op:cu256:m0:f1:h0:nb4:129x128", "k2:batch:cu256:m0:f1:h0:nb4:129x100,"
    job = {"box": 128, "spaces": 100, "fast": 1}
    small = {"box": 48, "spaces": 50, "fast": 1}
    keys = [k for k, in L.ask("op_key", [job, {**job, "init": 1500}, {**job, "spaces": 1500},
                                         small, {**small, "init": 200}])]
    keys += [k for k, in L.ask("batch_key", [job, {**job, "bounded": 1}])]
    assert len(set(keys)) == len(keys)
    assert old_op not in keys and old_batch not in keys
    # launches that do not differ share their line
    a, b = L.ask("op_key", [{**job, "spaces": 70}, {**job, "spaces": 128}])
    assert a == b


@pytest.mark.parametrize("skip", [{"table": 15000}, {"kernel": L.PAIR}, {"kernel": L.STAGED},
                                  {"count": 1}, {"tableGlobal": 1}])
@pytest.mark.parametrize("box", [8, 16, 32, 48, 100, 160, 224])
def test_exact_launches_spread_the_core(box, skip):
    """Where the centre of a volume is taken as cells by the brick kernels, a launch has wavefronts
    for them too, up to the GPU's: most of a small volume is cells (box 16: 728, and one brick)."""
    which, blocks, threads, _, _ = L.choices([{"box": box, "spaces": 100, **skip}])[0]
    assert which in (L.PAIR, L.STAGED)
    cells, bricks = (int(n) for n in L.ask("core", [{"box": box}])[0])
    waves = blocks * threads // 64
    assert waves >= min(max(cells, bricks), 256 * threads // 64) and blocks <= 256


def test_six_wide_fp32_kernels_keep_their_registers(metadata):
    """Kernels of six FP32 columns (radii from 2.75) with the table in LDS hold no registers in
    scratch memory, the exact brick kernels at most a few, which hold a row's pixels ahead; with two
    rows in flight they held up to 90 and took twice the time and more."""
    symbols = {c[-1] for c in L.choices(
        [{"box": box, "spaces": 1000, "radius": r, "batched": b, "fast": f, "kernel": k, "count": n}
         for box in (32, 64, 100, 200) for r in (2.8, 3.5) for b in (0, 1) for f in (0, 1)
         for k in (0, L.PAIR) for n in (0, 1)])}
    assert len(symbols) >= 10
    for symbol in symbols:
        exact_bricks = "16fr_insert_kernelILi0ELi0ELi6ELb0ELb0E" in symbol
        assert metadata[symbol][".vgpr_spill_count"] <= (24 if exact_bricks else 0), symbol


# (options, largest box of the small-problem kernel, spaces from which it takes that box)
CELL_RULES = [
    ({"radius": 1.2}, 104, 240), ({"radius": 1.5}, 104, 240), ({}, 86, 168),
    ({"radius": 2.5}, 120, 228), ({"radius": 3.6}, 120, 228), ({"fast": 1}, 104, 250),
    ({"fast": 1, "radius": 2.8}, 104, 250), ({"half": 1}, 114, 300),
    ({"half": 1, "radius": 2.8}, 96, 210), ({"evaluated": 1}, 120, 180), ({"nearest": 1}, 84, 160)]


@pytest.mark.parametrize("options,box,spaces", CELL_RULES)
def test_lines_of_the_small_problem_kernel(options, box, spaces):
    """Which launches run the small-problem kernel: boxes up to the line of the mode, radius and
    precision, from a number of spaces that grows with the box; no counting pass, named kernel or
    table beyond LDS."""
    case = {**options, "box": box, "spaces": spaces}
    others = [{**case, "box": box + 2, "spaces": 5000}, {**case, "spaces": spaces - 1},
              {**case, "count": 1}, {**case, "kernel": L.PAIR}, {**case, "batched": 1}]
    if not (options.get("evaluated") or options.get("nearest")):
        others += [{**case, "table": 11777}, {**case, "tableGlobal": 1}]
    got = [c[0] for c in L.choices([case, *others])]
    assert got[0] == L.CELLS and L.CELLS not in got[1:]


@pytest.mark.parametrize("fast", [0, 1])
def test_depth_scale_of_large_volumes_in_batches(fast):
    """Bricks of a batch's volumes above 165^3 are as thick as a plain operation's, whose heaviest
    brick a launch waits for, too; a bounded launch's are thicker."""
    for box in (166, 176, 208, 210, 256, 400):
        (batch, plain), (bounded, _) = L.ask("depth", [{"box": box, "fast": fast},
                                                       {"box": box, "fast": fast, "bounded": 1}])
        assert batch == plain and float(bounded) == 0.5
    assert L.ask("depth", [{"box": 160, "fast": fast}])[0][0] == "1"

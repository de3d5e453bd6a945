"""Launches at the limits of what a kernel holds or assumes, against the oracle."""
import numpy as np
import pytest

import launchtools
from frtools import problem, rel_l2, run_oracle, settings
from test_launch_rules import CELL_RULES
from umpalumpa_amd import fr as F

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n_table", [10747, 10748, 10751, 11776])
@pytest.mark.parametrize("strategy", [F.FR_EXACT, F.FR_FAST_MATH])
def test_batch_tables_around_the_carried_queues_limit(n_table, strategy):
    """A batch of FP32 jobs with tables up to the carried queues' limit (10,747 samples), beyond it
    (the per-pair kernel) and up to the largest a batch takes."""
    dev = torch.device("cuda:0")
    s = settings()
    jobs, ref = [], []
    table = F.fill_blob_table(n_table, F.fr_desc(17, 32, 9, 33, 9, n_table), s)
    d_table = torch.from_numpy(table).to(dev)  # the radius' table, of whatever box
    for box, n in ((32, 9), (48, 7)):
        fft, spaces, _, _ = problem(box, n, s, seed=box)
        jobs.append(F.BatchJob(torch.from_numpy(fft).to(dev),
                               torch.zeros((box + 1,) * 3, dtype=torch.complex64, device=dev),
                               torch.zeros((box + 1,) * 3, dtype=torch.float32, device=dev),
                               torch.from_numpy(spaces.view(np.uint8)).to(dev), s, d_table))
        ref.append(run_oracle(s, fft, spaces, table, box)[:2])
    b = F.FRBatch(0)
    b.plan(jobs, 5, strategy, graph=False)
    b.execute()
    b.synchronize()
    for job, (rv, rw) in zip(jobs, ref):
        v, w = job.volume.cpu().numpy(), job.weights.cpu().numpy()
        if strategy == F.FR_EXACT:
            assert v.tobytes() == rv.tobytes() and w.tobytes() == rw.tobytes()
        else:
            assert rel_l2(v, rv) <= 1e-5 and rel_l2(w, rw) <= 1e-5


def _beside_nan(box, n, s, **kw):
    """A problem whose odd slices, which no space names, hold NaN."""
    fft, spaces, desc, table = problem(box, 2 * n, s, **kw)
    keep = np.ascontiguousarray(spaces[spaces["projectionIndex"] % 2 == 0])
    fft[1::2] = np.complex64(complex(np.nan, np.nan))
    return fft, keep, desc, table


SLICES_BESIDE_NAN = [
    # table radius that does not slide, evaluated blobs, the widest boxes, slices below a box
    (30, F.FR_LOOKUP, 0.4), (30, F.FR_DYNAMIC, 1.9), (30, F.FR_LOOKUP, 3.2), (4, F.FR_LOOKUP, 1.9),
    (30, F.FR_DYNAMIC, 2.6), (130, F.FR_DYNAMIC, 1.9), (130, F.FR_LOOKUP, 0.4)]


@pytest.mark.parametrize("box,interp,radius", SLICES_BESIDE_NAN)
@pytest.mark.parametrize("kernel", [F.FR_KERNEL_AUTO, F.FR_KERNEL_PAIR])
def test_a_slice_beside_others_that_are_not_finite(box, interp, radius, kernel):
    """Candidate boxes that reach past a slice's last row take nothing of the next slice, which is
    NaN here and named by no space: the oracle's bits (exact), 1e-5 of them (fast math, FP16)."""
    from frtools import quantize_f16, run_hip
    s = settings(interp, radius=radius)
    fft, spaces, desc, table = _beside_nan(box, 9, s, seed=box)
    ov, ow, _ = run_oracle(s, fft, spaces, table, box)
    assert np.isfinite(ov.view(np.float32)).all() and ow.max() > 0
    sched = F.SchedParams(1.0, 1, 1, 0.5, kernel, 0, 0)
    v, w, _ = run_hip(s, fft, spaces, desc, table, box, sched=sched)
    assert v.tobytes() == ov.tobytes() and w.tobytes() == ow.tobytes()
    if interp != F.FR_LOOKUP:
        return
    v, w, _ = run_hip(s, fft, spaces, desc, table, box, strategy=F.FR_FAST_MATH, sched=sched)
    assert rel_l2(v, ov) <= 1e-5 and rel_l2(w, ow) <= 1e-5
    h, scales, deq = quantize_f16(np.where(np.isfinite(fft), fft, np.complex64(1)))
    h[1::2] = np.nan
    ov, ow, _ = run_oracle(s, deq, spaces, table, box)
    v, w, _ = run_hip(s, fft, spaces, desc, table, box, half=(h, scales), sched=sched)
    assert rel_l2(v, ov) <= 1e-5 and rel_l2(w, ow) <= 1e-5


@pytest.mark.parametrize("radius", [0.4, 1.9])
def test_a_batch_beside_slices_that_are_not_finite(radius):
    """The same through a batch of FP32 jobs (carried queues), slices of 3 x 4 pixels among them."""
    dev = torch.device("cuda:0")
    s = settings(radius=radius)
    jobs, ref = [], []
    for box in (4, 30):
        fft, spaces, _, table = _beside_nan(box, 9, s, seed=box)
        jobs.append(F.BatchJob(torch.from_numpy(fft).to(dev),
                               torch.zeros((box + 1,) * 3, dtype=torch.complex64, device=dev),
                               torch.zeros((box + 1,) * 3, dtype=torch.float32, device=dev),
                               torch.from_numpy(spaces.view(np.uint8)).to(dev), s,
                               torch.from_numpy(table).to(dev)))
        ref.append(run_oracle(s, fft, spaces, table, box)[:2])
    b = F.FRBatch(0)
    b.step(jobs, [0, 0], [j.n_spaces for j in jobs], F.FR_FAST_MATH)
    b.synchronize()
    for job, (rv, rw) in zip(jobs, ref):
        assert rel_l2(job.volume.cpu().numpy(), rv) <= 1e-5
        assert rel_l2(job.weights.cpu().numpy(), rw) <= 1e-5


@pytest.mark.parametrize("strategy", [F.FR_EXACT, F.FR_FAST_MATH])
def test_transforms_that_are_no_rotation(strategy):
    """A record's transform may be any matrix.  With its third row 1,500 times a rotation's, q.z
    rounds by hundredths at the slab's faces, and every voxel that passes the reference's rounded
    test has to be found: the oracle's number of updates, and under the exact strategy its bits."""
    from frtools import run_hip
    s = settings()
    box = 256
    fft, spaces, desc, table = problem(box, 200, s, seed=11)
    spaces["transformInv"][:, 2, :] *= np.float32(1500)
    ov, ow, updates = run_oracle(s, fft, spaces, table, box)
    v, w, n = run_hip(s, fft, spaces, desc, table, box, strategy=strategy, count=True)
    assert n == updates > 0
    if strategy == F.FR_EXACT:
        assert v.tobytes() == ov.tobytes() and w.tobytes() == ow.tobytes()
        v, w, _ = run_hip(s, fft, spaces, desc, table, box)
        assert v.tobytes() == ov.tobytes() and w.tobytes() == ow.tobytes()


def test_older_tuning_lines_are_not_used(tmp_path, monkeypatch):
    """A line that a build wrote in which its knobs meant other launches is no result for this one:
    the tuner times its candidates and writes a line of its own."""
    monkeypatch.setenv("UMPA_TUNING_DIR", str(tmp_path))
    dev = torch.device("cuda:0")
    s = settings()
    fft, spaces, desc, table = problem(48, 30, s)
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    path = tmp_path / "fr_tuning.txt"
    path.write_text(f"k2:op:cu{cus}:m0:f0:h0:nb4:49x32 0.5 0 1 0.5 1 1 0 0.1\n")
    op = F.FourierReconstruction(0)
    assert op.init(desc, s)
    d = [torch.from_numpy(a).to(dev) for a in (fft, spaces.view(np.uint8), table)]
    op.autotune(*d, use_cache=True)
    assert len(path.read_text().splitlines()) == 2


@pytest.mark.parametrize("options,box,spaces", CELL_RULES)
def test_volumes_on_either_side_of_the_small_problem_kernels_line(options, box, spaces):
    """The largest volume of the small-problem kernel in each mode, and the next box, which bricks
    take, with the fewest spaces that reach the rule."""
    from frtools import quantize_f16, run_hip
    evaluated, nearest = options.get("evaluated"), options.get("nearest")
    s = settings(F.FR_DYNAMIC if evaluated or nearest else F.FR_LOOKUP,
                 F.FR_FAST if nearest else F.FR_PRECISE, 15.0, options.get("radius", 1.9))
    for size, cells in ((box, True), (box + 2, False)):
        which = launchtools.choices([{**options, "box": size, "spaces": spaces}])[0][0]
        assert (which == launchtools.CELLS) == cells
        fft, sp, desc, table = problem(size, spaces, s, seed=size)
        if options.get("half"):
            h, scales, deq = quantize_f16(fft)
            ov, ow, _ = run_oracle(s, deq, sp, table, size)
            v, w, _ = run_hip(s, fft, sp, desc, table, size, half=(h, scales))
        else:
            ov, ow, _ = run_oracle(s, fft, sp, table, size)
            v, w, _ = run_hip(s, fft, sp, desc, table, size,
                              strategy=F.FR_FAST_MATH if options.get("fast") else F.FR_EXACT)
        if options.get("half") or options.get("fast"):
            assert rel_l2(v, ov) <= 1e-5 and rel_l2(w, ow) <= 1e-5
        else:
            assert v.tobytes() == ov.tobytes() and w.tobytes() == ow.tobytes()


@pytest.mark.parametrize("n_table", [10239, 10240, 10747, 10752, 11776])
@pytest.mark.parametrize("strategy", [F.FR_EXACT, F.FR_FAST_MATH])
def test_tables_across_the_brick_kernels_limits(n_table, strategy):
    """Tables on both sides of the staged and carried queues' limits, and the largest in LDS, in a
    volume that bricks take."""
    from frtools import run_hip
    s = settings()
    box, n = 124, 12
    which = launchtools.choices([{"box": box, "spaces": n, "table": n_table,
                                  "fast": int(strategy == F.FR_FAST_MATH)}])[0][0]
    limit, kernel = ((10751, launchtools.CARRY) if strategy == F.FR_FAST_MATH
                     else (10239, launchtools.STAGED))
    assert which == (kernel if n_table <= limit else launchtools.PAIR)
    fft, sp, _, _ = problem(box, n, s, seed=6)
    desc = F.fr_desc(box // 2 + 1, box, n, box + 1, len(sp), n_table)
    table = F.fill_blob_table(n_table, desc, s)
    ov, ow, _ = run_oracle(s, fft, sp, table, box)
    v, w, _ = run_hip(s, fft, sp, desc, table, box, strategy=strategy)
    if strategy == F.FR_EXACT:
        assert v.tobytes() == ov.tobytes() and w.tobytes() == ow.tobytes()
    else:
        assert rel_l2(v, ov) <= 1e-5 and rel_l2(w, ow) <= 1e-5


@pytest.mark.parametrize("half", [False, True])
def test_every_fast_math_candidate_on_bricks(half):
    """The fast-math tuner's knob sets in a volume whose default kernel runs schedules."""
    from frtools import quantize_f16, run_hip
    s = settings()
    box, n = 124, 30
    fft, sp, desc, table = problem(box, n, s, seed=43)
    h = None
    if half:
        *h, fft = quantize_f16(fft)
    ov, ow, _ = run_oracle(s, fft, sp, table, box)
    for p in F.tuning_candidates(F.FR_FAST_MATH):
        v, w, _ = run_hip(s, fft, sp, desc, table, box, strategy=F.FR_FAST_MATH, half=h, sched=p)
        assert rel_l2(v, ov) <= 1e-5 and rel_l2(w, ow) <= 1e-5, p.as_tuple()


@pytest.mark.parametrize("typ", [F.FR_PRECISE, F.FR_FAST])
@pytest.mark.parametrize("box,n", [(84, 160), (84, 59), (86, 160)])
def test_shared_cells_without_a_table(box, n, typ):
    """Shared central cells up to 85^3 where no table is read, and beyond, from 60 spaces on."""
    from frtools import run_hip
    s = settings(F.FR_DYNAMIC, typ, 15.0, 1.9)
    fft, sp, desc, table = problem(box, n, s, seed=n)
    ov, ow, _ = run_oracle(s, fft, sp, table, box)
    v, w, _ = run_hip(s, fft, sp, desc, table, box)
    assert v.tobytes() == ov.tobytes() and w.tobytes() == ow.tobytes()

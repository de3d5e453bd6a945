"""The small-problem insertion kernel (cells of 2 x 2 x 2 voxels, eight spaces at a time) where it
can go wrong: volumes at and around the edges of its cells, blocks and size rule, numbers of
spaces around its steps of 8, its queue entries of 64 and its tiles of 1,024, every mode and
footprint.  Exact strategy: bit-identical to the oracle; fast math and FP16: 1e-5 relative L2."""
import numpy as np
import pytest

import pyoracle
from frtools import (problem, quantize_f16, rel_l2, run_hip, run_oracle, settings,
                     synthetic_slices)
from umpalumpa_amd import fr as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box,n", [(2, 3), (6, 1), (8, 7), (14, 8), (16, 9), (30, 64), (34, 65),
                                   (22, 1023), (20, 1025), (12, 2100), (116, 12), (118, 12)])
def test_sizes(box, n):
    s = settings()
    fft, spaces, desc, table = problem(box, n, s, seed=box + n)
    ov, ow, _ = run_oracle(s, fft, spaces, table, box)
    v, w, _ = run_hip(s, fft, spaces, desc, table, box)
    assert v.tobytes() == ov.tobytes() and w.tobytes() == ow.tobytes()
    v, w, _ = run_hip(s, fft, spaces, desc, table, box, strategy=F.FR_FAST_MATH)
    assert rel_l2(v, ov) <= 1e-5 and rel_l2(w, ow) <= 1e-5
    h, scales, deq = quantize_f16(fft)
    ov, ow, _ = run_oracle(s, deq, spaces, table, box)
    v, w, _ = run_hip(s, fft, spaces, desc, table, box, half=(h, scales))
    assert rel_l2(v, ov) <= 1e-5 and rel_l2(w, ow) <= 1e-5


@pytest.mark.parametrize("box,n", [(128, 256), (144, 256)])
def test_many_spaces_rule(box, n):
    s = settings(radius=1.2)
    fft, spaces, desc, table = problem(box, n, s, seed=4)
    ov, ow, _ = run_oracle(s, fft, spaces, table, box)
    v, w, _ = run_hip(s, fft, spaces, desc, table, box)
    assert v.tobytes() == ov.tobytes() and w.tobytes() == ow.tobytes()


@pytest.mark.parametrize("interp,typ,alpha,radius", [
    (F.FR_LOOKUP, F.FR_PRECISE, 15.0, 0.4), (F.FR_LOOKUP, F.FR_PRECISE, 15.0, 1.0),
    (F.FR_LOOKUP, F.FR_PRECISE, 15.0, 2.2), (F.FR_LOOKUP, F.FR_PRECISE, 15.0, 2.5),
    (F.FR_LOOKUP, F.FR_PRECISE, 15.0, 2.9), (F.FR_LOOKUP, F.FR_PRECISE, 15.0, 3.2),
    (F.FR_DYNAMIC, F.FR_PRECISE, 15.0, 1.9), (F.FR_DYNAMIC, F.FR_PRECISE, 12.0, 2.5),
    (F.FR_DYNAMIC, F.FR_FAST, 15.0, 1.9)])
@pytest.mark.parametrize("box", [10, 42])
def test_modes_and_radii(box, interp, typ, alpha, radius):
    s = settings(interp, typ, alpha, radius)
    sym = [np.eye(3), np.diag([-1.0, -1.0, 1.0])]
    fft, spaces, desc, table = problem(box, 21, s, seed=8, symmetries=sym)
    spaces["weight"][::3] = 0.5
    ov, ow, _ = run_oracle(s, fft, spaces, table, box)
    v, w, _ = run_hip(s, fft, spaces, desc, table, box)
    assert v.tobytes() == ov.tobytes() and w.tobytes() == ow.tobytes()


def test_accumulates_in_order_and_leaves_the_rest():
    """Chunks into a volume that holds values, -0 among them: touched voxels take the oracle's
    bits, the others keep their own; slices of another size than the volume's half plane, a
    space naming no slice."""
    box, n = 26, 40
    s = settings()
    fft = synthetic_slices(box, n, 3)[:, :, :9]
    spaces = F.traverse_spaces(pyoracle.uniform_rotations(n, 6), box, s)
    spaces["projectionIndex"][5] = n + 3
    desc = F.fr_desc(9, box, n, box + 1, n, 10000)
    table = F.fill_blob_table(10000, desc, s)
    rng = np.random.default_rng(1)
    v0 = rng.standard_normal((box + 1,) * 3 + (2,)).astype(np.float32)
    v0[rng.random(v0.shape) < 0.3] = -0.0
    v0 = np.ascontiguousarray(v0).view(np.complex64)[..., 0]
    w0 = rng.random((box + 1,) * 3).astype(np.float32)
    keep = np.delete(np.arange(n), 5)
    ov, ow, _ = run_oracle(s, fft, np.ascontiguousarray(spaces[keep]), table, box, v0, w0)
    v, w, _ = run_hip(s, np.ascontiguousarray(fft), spaces, desc, table, box, chunks=3, volume=v0,
                      weights=w0)
    assert v.tobytes() == ov.tobytes() and w.tobytes() == ow.tobytes()


@pytest.mark.parametrize("box", [104, 130, 160, 162, 198, 224, 226])
@pytest.mark.parametrize("kernel", [F.FR_KERNEL_AUTO, F.FR_KERNEL_PAIR])
def test_core_of_larger_volumes(box, kernel):
    """The exact strategy takes the centre of volumes up to 225^3 as cells: both exact kernels,
    table in LDS and global, the update count, boxes around the lines of the core's radius."""
    s = settings(radius=1.5 if box % 4 else 1.9)
    fft, spaces, desc, table = problem(box, 11, s, seed=box)
    ov, ow, updates = run_oracle(s, fft, spaces, table, box)
    sched = F.SchedParams(1.0, 1, 1, 0.5, kernel, 1 if box == 162 else 0, 0)
    for count in (False, True):
        v, w, n = run_hip(s, fft, spaces, desc, table, box, sched=sched, count=count)
        assert v.tobytes() == ov.tobytes() and w.tobytes() == ow.tobytes()
    assert n == updates


@pytest.mark.parametrize("typ", [F.FR_PRECISE, F.FR_FAST])
def test_core_without_table(typ):
    s = settings(F.FR_DYNAMIC, typ, 15.0, 1.9)
    fft, spaces, desc, table = problem(134, 9, s, seed=2)
    ov, ow, _ = run_oracle(s, fft, spaces, table, 134)
    v, w, _ = run_hip(s, fft, spaces, desc, table, 134)
    assert v.tobytes() == ov.tobytes() and w.tobytes() == ow.tobytes()


def test_no_core_where_slices_exceed_one_resource():
    """A chunk of more than 2 GiB of slices (13,400 of 101 x 200) gives the small chunk's bits."""
    import torch
    box = 200
    s = settings()
    fft, spaces, _, table = problem(box, 3, s, seed=17)
    dev = torch.device("cuda:0")
    d_tab = torch.from_numpy(table).to(dev)
    d_sp = torch.from_numpy(np.ascontiguousarray(spaces).view(np.uint8)).to(dev)
    big = torch.zeros((13400,) + fft.shape[1:], dtype=torch.complex64, device=dev)
    big[:3] = torch.from_numpy(np.ascontiguousarray(fft)).to(dev)
    out = []
    for buf in (big[:3], big):
        desc = F.fr_desc(fft.shape[2], fft.shape[1], buf.shape[0], box + 1, len(spaces), table.size)
        op = F.FourierReconstruction(0)
        assert op.init(desc, s)
        vol = torch.zeros((box + 1,) * 3, dtype=torch.complex64, device=dev)
        wts = torch.zeros((box + 1,) * 3, dtype=torch.float32, device=dev)
        assert op.execute(buf, vol, wts, d_sp, d_tab)
        op.synchronize()
        out.append((vol.cpu().numpy().tobytes(), wts.cpu().numpy().tobytes()))
    assert out[0] == out[1]


@pytest.mark.parametrize("items", [1, 2, 5, 1000])
@pytest.mark.parametrize("strategy", [F.FR_EXACT, F.FR_FAST_MATH])
def test_dealt_items_cover_every_brick(items, strategy):
    """Bounded launches deal their items out by workgroup: sizes around one group of workgroups,
    a last group that is short, fewer items than a workgroup's share."""
    import torch
    dev = torch.device("cuda:0")
    s = settings()
    jobs, ref = [], []
    for box, n in ((8, 5), (66, 6), (136, 4)):
        fft, spaces, desc, table = problem(box, n, s, seed=box)
        jobs.append(F.BatchJob(torch.from_numpy(fft).to(dev),
                               torch.zeros((box + 1,) * 3, dtype=torch.complex64, device=dev),
                               torch.zeros((box + 1,) * 3, dtype=torch.float32, device=dev),
                               torch.from_numpy(spaces.view(np.uint8)).to(dev), s,
                               torch.from_numpy(table).to(dev)))
        ref.append(run_oracle(s, fft, spaces, table, box)[:2])
    for chosen in ([0], [0, 1, 2]):
        b = F.FRBatch(0)
        b.set_wave_items(items)
        for k in chosen:
            jobs[k].volume.zero_()
            jobs[k].weights.zero_()
        part = [jobs[k] for k in chosen]
        b.step(part, [0] * len(part), [j.n_spaces for j in part], strategy)
        b.synchronize()
        for k in chosen:
            v, w = jobs[k].volume.cpu().numpy(), jobs[k].weights.cpu().numpy()
            if strategy == F.FR_EXACT:
                assert v.tobytes() == ref[k][0].tobytes() and w.tobytes() == ref[k][1].tobytes()
            else:
                assert rel_l2(v, ref[k][0]) <= 1e-5 and rel_l2(w, ref[k][1]) <= 1e-5


@pytest.mark.parametrize("interp,typ", [(F.FR_LOOKUP, F.FR_PRECISE), (F.FR_DYNAMIC, F.FR_PRECISE),
                                        (F.FR_DYNAMIC, F.FR_FAST)])
@pytest.mark.parametrize("box,n", [(2, 60), (4, 61), (10, 95), (56, 97), (58, 64), (16, 1057)])
def test_shared_cells(box, n, interp, typ):
    """Cells that four wavefronts share (from 60 spaces on, volumes up to 57^3, or 85^3 without a
    table): cells outside the volume, rounds of 32 spaces with a remainder, several tiles; the same
    operation with fewer spaces than a round, and onto values it holds."""
    s = settings(interp, typ, 15.0, 1.9)
    fft, spaces, desc, table = problem(box, n, s, seed=box + n)
    spaces["weight"][::3] = 0.5
    ov, ow, _ = run_oracle(s, fft, spaces, table, box)
    for chunks in (1, 5):
        v, w, _ = run_hip(s, fft, spaces, desc, table, box, chunks=chunks)
        assert v.tobytes() == ov.tobytes() and w.tobytes() == ow.tobytes()
    if interp == F.FR_LOOKUP:
        v, w, _ = run_hip(s, fft, spaces, desc, table, box, strategy=F.FR_FAST_MATH)
        assert rel_l2(v, ov) <= 1e-5 and rel_l2(w, ow) <= 1e-5

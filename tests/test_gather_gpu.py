"""The insertion's gather where its candidate boxes are tight (r = 1.5 and 2.5: boxes of 2r
columns), at the positions and slice sizes where one more column, the box's slide or a remainder
could go wrong.  Exact strategy: bit-identical to the oracle; fast math and FP16 slices: the
strategy's 1e-5 relative L2."""
import numpy as np
import pytest

import pyoracle
from frtools import quantize_f16, rel_l2, run_hip, run_oracle, settings, synthetic_slices
from umpalumpa_amd import fr as F

pytestmark = pytest.mark.gpu


def _half_step_rotations():
    """Orientations whose entries are multiples of 1/2 as floats: voxels land on whole and half
    pixels, so that q - r and q + r are both whole numbers for r = 1.5 and 2.5."""
    out = [np.eye(3)]
    for axis in range(3):
        m = np.zeros((3, 3))
        a, b = [k for k in range(3) if k != axis]
        m[axis, axis] = 1.0
        m[a, b], m[b, a] = -1.0, 1.0
        out.append(m)
        h = np.eye(3)  # 60 degrees: cosine 1/2, sine irrational
        c, s = 0.5, 3.0 ** 0.5 / 2
        h[a, a], h[a, b], h[b, a], h[b, b] = c, -s, s, c
        out.append(h)
    return np.array(out)


@pytest.mark.parametrize("radius", [1.5, 2.5, 1.5 - 4e-7, 2.5 + 4e-7])
@pytest.mark.parametrize("box", [8, 30, 64])
def test_tight_boxes_at_pixel_ties(box, radius):
    s = settings(radius=radius)
    rots = np.concatenate([_half_step_rotations(), pyoracle.uniform_rotations(9, 3)])
    fft = synthetic_slices(box, len(rots), 5)
    spaces = F.traverse_spaces(rots, box, s, weight=0.75)
    desc = F.fr_desc(box // 2 + 1, box, len(rots), box + 1, len(spaces), 10000)
    table = F.fill_blob_table(10000, desc, s)
    ov, ow, updates = run_oracle(s, fft, spaces, table, box)
    v, w, _ = run_hip(s, fft, spaces, desc, table, box)
    assert v.tobytes() == ov.tobytes() and w.tobytes() == ow.tobytes()
    v, w, n = run_hip(s, fft, spaces, desc, table, box, count=True)
    assert v.tobytes() == ov.tobytes() and w.tobytes() == ow.tobytes() and n == updates
    v, w, _ = run_hip(s, fft, spaces, desc, table, box, strategy=F.FR_FAST_MATH)
    assert rel_l2(v, ov) <= 1e-5 and rel_l2(w, ow) <= 1e-5
    h, scales, deq = quantize_f16(fft)
    ov, ow, _ = run_oracle(s, deq, spaces, table, box)
    v, w, _ = run_hip(s, fft, spaces, desc, table, box, half=(h, scales))
    assert rel_l2(v, ov) <= 1e-5 and rel_l2(w, ow) <= 1e-5


@pytest.mark.parametrize("alpha,order", [(15.0, 0), (16.0, 2)])
@pytest.mark.parametrize("radius", [0.3, 1.9, 2.0, 2.6])
@pytest.mark.parametrize("box,n", [(6, 9), (30, 13), (130, 3)])
def test_evaluated_blobs(box, n, radius, alpha, order):
    """Blob values computed for a wavefront's candidates together: no candidate or few inside
    (r = 0.3), boxes with a fifth column (r = 2.0 at ties, 2.6 always: the general loop beside
    the box in one wavefront), slices narrower than a box, weights other than 1.  Small boxes
    take cells, the counting pass and box 130 bricks (its core: cells)."""
    s = settings(F.FR_DYNAMIC, F.FR_PRECISE, alpha, radius, order)
    rots = np.concatenate([_half_step_rotations()[:2], pyoracle.uniform_rotations(n, 3)])
    fft = synthetic_slices(box, len(rots), 5)
    spaces = F.traverse_spaces(rots, box, s, weight=0.75)
    spaces["weight"][::2] = 1.0
    desc = F.fr_desc(box // 2 + 1, box, len(rots), box + 1, len(spaces), 0)
    ov, ow, updates = run_oracle(s, fft, spaces, None, box)
    v, w, _ = run_hip(s, fft, spaces, desc, None, box)
    assert np.array_equal(v, ov, equal_nan=True) and np.array_equal(w, ow, equal_nan=True)
    v, w, got = run_hip(s, fft, spaces, desc, None, box, count=True)
    assert np.array_equal(v, ov, equal_nan=True) and np.array_equal(w, ow, equal_nan=True)
    assert got == updates

"""Launches at the limits of what a kernel holds or assumes, against the oracle."""
import numpy as np
import pytest

from frtools import problem, rel_l2, run_oracle, settings
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

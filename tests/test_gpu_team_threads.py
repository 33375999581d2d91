"""One-launch solves of the same kernel with different LDS sizes from several threads at once."""

import threading

import pytest
import torch

from tests.test_gpu_team_streams import Job

pytestmark = pytest.mark.gpu


def test_sizes_of_one_kernel_in_threads(ctx):
    print('LDS sizes in threads', flush=True)
    jobs = [Job('tri_elastic', size) for size in [(3, 2), (15, 7), (20, 10), (15, 15)]]  # one workgroup each
    want = [job.solve(tol=1e-9) for job in jobs]
    wrong = []

    def run(job, ref):
        torch.cuda.set_device(0)
        for _ in range(50):
            x, info = job.solve(tol=1e-9)
            if info['path'] != ref[1]['path'] or not torch.equal(x, ref[0]):
                wrong.append(info)

    threads = [threading.Thread(target=run, args=a) for a in zip(jobs, want)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong

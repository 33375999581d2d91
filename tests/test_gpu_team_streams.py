"""One-launch solves on several streams at once: a solve of one workgroup does not wait for another stream's, a
larger one finds the device taken and runs by the launched kernels, and all give the bits they give alone."""

import threading
import time

import pytest
import torch

from finite_elements_amd import _hip
from finite_elements_amd.device import Context
from finite_elements_amd.system import FESystem
from tests.test_gpu_team import _problem

pytestmark = pytest.mark.gpu

ONE_LAUNCH, LAUNCHED = _hip.FE_PCG_ONE_LAUNCH, _hip.FE_PCG_LAUNCHED


class Job:
    """A system, its solver and its own handle and stream."""

    def __init__(self, kind, size, seed=0):
        base, fixed, rng = _problem(kind, size, seed=seed)
        self.ctx = Context(0, torch.cuda.Stream())
        with torch.cuda.stream(self.ctx.stream):
            ne = base.n_elem
            s = FESystem(kind, base._coords, base._conn, {'E': torch.ones(ne).numpy(), 'nu': 0.3, 'thickness': 1.0},
                         plane_mode=base.mesh.plane_mode, ctx=self.ctx)
            mask, g = s.dirichlet(fixed)
            KD, self.b = s.prepare(s.stiffness_bsr(), mask, g, self.ctx.tensor(rng.standard_normal(s.n)))
            self.solver = s.solver(KD, 'jacobi', 'fp64')
        self.ctx.stream.synchronize()

    def solve(self, **kw):
        with torch.cuda.stream(self.ctx.stream):
            x, info = self.solver.solve(self.b, **kw)
            self.ctx.stream.synchronize()
        return x, info

    def start(self, **kw):
        def run():
            torch.cuda.set_device(0)
            self.out = self.solve(**kw)
        self.thread = threading.Thread(target=run)
        self.thread.start()


#: no residual is below the tolerance: tens of thousands of iterations of about 7 us
LONG = {'tol': 1e-250, 'max_iter': 60000}


def test_one_workgroup_beside_a_long_solve(ctx):
    print('one workgroup beside a long solve', flush=True)
    long, small = Job('tet_elastic', 13), Job('tri_elastic', (16, 6))
    alone = small.solve(tol=1e-9)
    long.start(**LONG)
    time.sleep(0.05)
    x, info = small.solve(tol=1e-9)
    beside = long.thread.is_alive()
    long.thread.join()
    assert info['path'] == ONE_LAUNCH and torch.equal(x, alone[0])
    assert beside, 'the small solve waited for the long one'


def test_many_workgroups_beside_long_solves(ctx):
    print('many workgroups beside long solves', flush=True)
    longs, other = [Job('tet_elastic', 13, seed=k) for k in range(3)], Job('tet_elastic', 7)
    alone = other.solve(tol=1e-9)
    assert alone[1]['path'] == ONE_LAUNCH
    for job in longs:
        job.start(**LONG)
    time.sleep(0.05)
    x, info = other.solve(tol=1e-9)
    beside = all(job.thread.is_alive() for job in longs)
    for job in longs:
        job.thread.join()
    assert beside and info['path'] == LAUNCHED and torch.equal(x, alone[0])
    x, info = other.solve(tol=1e-9)
    assert info['path'] == ONE_LAUNCH and torch.equal(x, alone[0])


def test_bits_on_many_streams(ctx):
    print('bits on many streams', flush=True)
    jobs = [Job(kind, size, seed) for seed, (kind, size) in enumerate(
        [('tri_elastic', (16, 6)), ('tri_elastic', (40, 10)), ('tet_elastic', 7), ('tet_elastic', 13)] * 2)]
    alone = [job.solve(tol=1e-9) for job in jobs]
    for _ in range(3):
        for job in jobs:
            job.start(tol=1e-9)
        for job in jobs:
            job.thread.join()
        for job, want in zip(jobs, alone):
            assert job.out[1]['iterations'] == want[1]['iterations'] and torch.equal(job.out[0], want[0])

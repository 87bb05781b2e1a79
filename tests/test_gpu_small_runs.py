"""Runs of 4,097 to 16,384 spheres (row resort with the row-split collide, or
the radix sort on grids outside the resort's rule) against the oracle bit for
bit: runs and updates in turn, both radius modes, grids on both sides of the
rule's edges."""
from __future__ import annotations

import os

import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_parity import _compare_system

pytestmark = pytest.mark.gpu

R = 1.0 / 64.0


@pytest.fixture(scope="module", autouse=True)
def _oracle_threads():
    orc.set_threads(max(1, min(16, os.cpu_count() or 1)))
    yield
    orc.set_threads(1)


# 16 and 64 rows (n above and below 256 per row), 2^18 rows and twice that
@pytest.mark.parametrize("poly", [False, True])
@pytest.mark.parametrize("n,grid", [
    (4097, (64, 64, 64)), (9001, (32, 32, 32)), (16384, (64, 64, 64)), (16384, (64, 64, 16)),
    (16384, (8, 8, 8)), (4096 + 255, (16, 4, 4)), (16383, (64, 8, 8)), (5000, (4, 512, 512)),
    (5000, (4, 1024, 512))])
def test_small_runs_and_updates_match_oracle(gpu_ctx, n, grid, poly):
    from fullc0ntact_amd import ParticleSystem, make_params
    print(n, grid, poly, flush=True)
    rng = np.random.default_rng(n + grid[1])
    pos = np.ones((n, 4), np.float32)
    pos[:, :3] = rng.uniform(-0.95, 0.95, (n, 3))
    m = 200  # a pile that moves as a whole
    pos[:m, :3] = rng.uniform(-0.5, 0.5, 3) + rng.normal(0.0, 0.6 * R, (m, 3))
    if poly:
        pos[:, 3] = rng.uniform(0.6 * R, R, n)
    vel = np.zeros((n, 4), np.float32)
    vel[:, :3] = rng.uniform(-0.01, 0.01, (n, 3))
    P = make_params(n, grid[0], R, gridSize=grid, numCells=int(np.prod(grid)))
    ps = ParticleSystem(n, grid, context=gpu_ctx)
    ps.m_params = P
    ps.setPolydisperse(poly)
    ps.setArray(ps.POSITION, pos, 0, n)
    ps.setArray(ps.VELOCITY, vel, 0, n)
    st = orc.State(pos, vel, P.numCells)
    OP = orc.params_from(P)
    for run, steps in ((True, 4), (False, 1), (True, 2), (True, 10)):
        if run:
            ps.run(0.5, steps)
        else:
            ps.update(0.5)
        for _ in range(steps):
            orc.update_ex(st, 0.5, OP, None, poly=poly)
        _compare_system(ps, st)
    ps.close()

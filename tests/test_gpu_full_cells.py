"""The row-split collide where cells hold many spheres: rows whose cells are
full, empty or hold the sphere alone in every order, against the oracle bit for
bit."""
from __future__ import annotations

import os

import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_parity import _compare_system

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _oracle_threads():
    orc.set_threads(max(1, min(16, os.cpu_count() or 1)))
    yield
    orc.set_threads(1)


def cells_along_x(grid, counts, rng):
    """counts[i] spheres in the i-th cell of one row of cells."""
    edge = 2.0 / grid
    x = np.repeat(np.arange(len(counts)), counts)
    at = np.stack([x, np.full_like(x, grid // 2), np.full_like(x, grid // 2)], 1)
    return -1.0 + edge * (at + 0.5 + rng.uniform(-0.45, 0.45, at.shape))


@pytest.mark.parametrize("poly", [False, True])
@pytest.mark.parametrize("n", [700, 4096, 6000])
def test_rows_of_full_cells(gpu_ctx, n, poly):
    from fullc0ntact_amd import ParticleSystem, make_params
    grid, r = 32, 1.0 / 32.0
    rng = np.random.default_rng(n + poly)
    # every pattern of empty, lone and full neighbours, 0-9 spheres a cell
    counts = np.concatenate([rng.integers(0, 10, 8), [0, 5, 0, 0, 7, 1, 4, 4, 1, 3, 0, 8, 1, 0, 0]])
    full = cells_along_x(grid, counts, rng)
    xyz = np.concatenate([full, rng.uniform(-0.95, 0.95, (n - len(full), 3))])
    pos = np.ones((n, 4), np.float32)
    pos[:, :3] = rng.permutation(xyz)
    if poly:
        pos[:, 3] = rng.uniform(0.3 * r, r, n)
    vel = np.zeros((n, 4), np.float32)
    vel[:, :3] = rng.uniform(-0.01, 0.01, (n, 3))
    P = make_params(n, grid, r)
    ps = ParticleSystem(n, (grid,) * 3, context=gpu_ctx)
    ps.m_params = P
    ps.setPolydisperse(poly)
    ps.setArray(ps.POSITION, pos, 0, n)
    ps.setArray(ps.VELOCITY, vel, 0, n)
    st = orc.State(pos, vel, P.numCells)
    print(n, poly, flush=True)
    ps.update(0.5)
    orc.update_ex(st, 0.5, orc.params_from(P), None, poly=poly)
    _compare_system(ps, st)
    ps.run(0.5, 3)
    for _ in range(3):
        orc.update_ex(st, 0.5, orc.params_from(P), None, poly=poly)
    _compare_system(ps, st)
    ps.close()


@pytest.mark.parametrize("poly", [False, True])
@pytest.mark.parametrize("mean", [32, 50, 180])
def test_long_rows_of_cells(gpu_ctx, mean, poly):
    """Rows about and beyond the 96 candidates from which a wave may take them
    cell by cell, even, uneven and with gaps, in one launch."""
    from fullc0ntact_amd import ParticleSystem, make_params
    grid, r = 16, 1.0 / 16.0
    rng = np.random.default_rng(mean + poly)
    even = np.full(6, mean) + rng.integers(-1, 2, 6)
    counts = np.concatenate([even, [0, 3 * mean, 0, 0, 96, 1, 0, mean, 2 * mean, 5]])
    xyz = cells_along_x(grid, counts, rng)
    side = rng.uniform((-0.9, 0.4, 0.4), (0.9, 0.6, 0.6), (3 * mean, 3))
    xyz = np.concatenate([xyz, side, rng.uniform(-0.95, 0.95, (300, 3))])
    n = len(xyz)
    pos = np.ones((n, 4), np.float32)
    pos[:, :3] = rng.permutation(xyz)
    if poly:
        pos[:, 3] = rng.uniform(0.3 * r, r, n)
    vel = np.zeros((n, 4), np.float32)
    vel[:, :3] = rng.uniform(-0.01, 0.01, (n, 3))
    P = make_params(n, grid, r)
    ps = ParticleSystem(n, (grid,) * 3, context=gpu_ctx)
    ps.m_params = P
    ps.setPolydisperse(poly)
    ps.setArray(ps.POSITION, pos, 0, n)
    ps.setArray(ps.VELOCITY, vel, 0, n)
    st = orc.State(pos, vel, P.numCells)
    print(n, poly, flush=True)
    for _ in range(2):
        ps.update(0.01)
        orc.update_ex(st, 0.01, orc.params_from(P), None, poly=poly)
        _compare_system(ps, st)
    ps.close()

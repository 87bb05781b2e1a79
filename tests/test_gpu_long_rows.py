"""Row resort of rows beyond its LDS (768 members), and of rows all of whose
spheres move, against the oracle bit for bit: full cells on both sides of the
sizes that the parts of a row take together, one by one and by counting, rows
of more than 256 cells, small systems and larger ones."""
from __future__ import annotations

import os

import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_parity import _compare_system

pytestmark = pytest.mark.gpu

EDGE = 1.0 / 32.0


@pytest.fixture(scope="module", autouse=True)
def _oracle_threads():
    orc.set_threads(max(1, min(16, os.cpu_count() or 1)))
    yield
    orc.set_threads(1)


def in_cells(cells, rng):
    """A sphere in each of the cells (n,3), none near its faces."""
    return -1.0 + EDGE * (np.asarray(cells) + 0.5 + rng.uniform(-0.3, 0.3, (len(cells), 3)))


def row_state(kind, rng):
    """Cells of the spheres that stand in long rows (row y = 40, z = 20..27)."""
    if kind == "one row":
        return [(x, 40, 20) for x in rng.integers(2, 62, 3000)]
    if kind == "eight rows":
        return [(x, 40, 20 + i % 8) for i, x in enumerate(rng.integers(2, 62, 8 * 900))]
    if kind == "768 and 769":
        return [(2 + i % 60, 40, 20) for i in range(768)] + [(2 + i % 60, 40, 24) for i in range(769)]
    if kind == "full cells":
        return [(x, 40, 20) for x, k in ((5, 384), (9, 385), (10, 768), (20, 769), (30, 40),
                                         (31, 1), (40, 300)) for _ in range(k)]
    assert kind == "one cell"
    return [(30, 40, 20)] * 2000


# moving: cells a step in x (every sphere of the rows), in y, or slowly
@pytest.mark.parametrize("move", ["slow", "along", "across"])
@pytest.mark.parametrize("kind", ["one row", "eight rows", "768 and 769", "full cells", "one cell"])
def test_long_rows(gpu_ctx, kind, move):
    run_state(gpu_ctx, kind, move, 9000, (64, 64, 64))


@pytest.mark.parametrize("kind", ["one row", "full cells"])
def test_long_rows_of_larger_systems(gpu_ctx, kind):
    run_state(gpu_ctx, kind, "along", 36000, (64, 64, 64))


@pytest.mark.parametrize("kind", ["one row", "full cells", "one cell"])
def test_rows_of_many_cells(gpu_ctx, kind):
    """1,024 cells a row: four to a range, the walls within the first 64."""
    run_state(gpu_ctx, kind, "along", 9000, (1024, 64, 64))


def run_state(ctx, kind, move, n, grid):
    from fullc0ntact_amd import ParticleSystem, make_params
    print(kind, move, n, grid, flush=True)
    rng = np.random.default_rng(len(kind) + n)
    rows = in_cells(row_state(kind, rng), rng)
    m = len(rows)
    pos = np.ones((n, 4), np.float32)
    pos[:, :3] = np.concatenate([rows, rng.uniform(-0.95, 0.95, (n - m, 3))])
    vel = np.zeros((n, 4), np.float32)
    vel[:, :3] = rng.uniform(-0.002, 0.002, (n, 3))
    if move != "slow":
        vel[:m, 0 if move == "along" else 1] = EDGE / 0.5
    perm = rng.permutation(n)
    pos, vel = pos[perm], vel[perm]
    # no pair forces: the piles stay together
    P = make_params(n, grid[0], EDGE / 2, gridSize=grid, numCells=int(np.prod(grid)), spring=0.0,
                    damping=0.0, shear=0.0)
    ps = ParticleSystem(n, grid, context=ctx)
    ps.m_params = P
    ps.setArray(ps.POSITION, pos, 0, n)
    ps.setArray(ps.VELOCITY, vel, 0, n)
    st = orc.State(pos, vel, P.numCells)
    ps.run(0.5, 5)
    for _ in range(5):
        st.update(0.5, orc.params_from(P))
    _compare_system(ps, st)
    ps.close()

"""The row-range collide with one radius above the row-split kernel's range:
the walls' wrapped cells, caller-owned arrays, piles that move as a whole and
lists that overflow, against the oracle bit for bit; and both sides of the
line between the two kernels."""
from __future__ import annotations

import os

import numpy as np
import pytest

import test_gpu_wall_cells as walls
from oracle import oracle as orc
from test_gpu_parity import Stages, _compare_system, bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _oracle_threads():
    orc.set_threads(max(1, min(16, os.cpu_count() or 1)))
    yield
    orc.set_threads(1)


@pytest.fixture
def many(monkeypatch):
    monkeypatch.setattr(walls, "N", 40000)


@pytest.mark.parametrize("grid", [(32, 32, 32), (64, 32, 64), (16, 16, 16)])
def test_at_the_walls(gpu_ctx, many, grid):
    walls.test_system_at_the_walls(gpu_ctx, grid)


@pytest.mark.parametrize("outside", [False, True])
def test_through_the_wrap(gpu_ctx, many, outside):
    walls.test_stages_through_the_wrap(gpu_ctx, outside)


@pytest.mark.parametrize("pile", [65, 700])
def test_moving_piles(gpu_ctx, many, pile):
    walls.test_piles_that_move_as_a_whole(gpu_ctx, pile)


@pytest.mark.parametrize("loose", [36000, 30000 - 2700])
def test_overflowing_lists(gpu_ctx, loose):
    from fullc0ntact_amd import ParticleSystem, make_params
    grid, r = 64, 1.0 / 64.0
    rng = np.random.default_rng(45)
    parts = [rng.uniform(-0.95, 0.95, (loose, 3))]
    parts += [rng.uniform(-0.9, 0.9, 3) + rng.normal(scale=0.6 * r, size=(45, 3))
              for _ in range(60)]
    xyz = rng.permutation(np.concatenate(parts))
    n = len(xyz)
    pos = np.ones((n, 4), np.float32)
    pos[:, :3] = np.clip(xyz, -1 + r, 1 - r)
    vel = np.zeros((n, 4), np.float32)
    vel[:, :3] = rng.uniform(-0.01, 0.01, (n, 3))
    P = make_params(n, grid, r)
    ps = ParticleSystem(n, (grid,) * 3, context=gpu_ctx)
    ps.m_params = P
    ps.setArray(ps.POSITION, pos, 0, n)
    ps.setArray(ps.VELOCITY, vel, 0, n)
    st = orc.State(pos, vel, P.numCells)
    print(n, flush=True)
    ps.update(0.5)
    ps.run(0.5, 6)
    for _ in range(7):
        st.update(0.5, orc.params_from(P))
    _compare_system(ps, st)
    ps.close()


@pytest.mark.parametrize("n", [32768, 32769])
def test_either_side_of_the_line(gpu_ctx, n):
    from fullc0ntact_amd import ParticleSystem, make_params
    rng = np.random.default_rng(n)
    pos = np.ones((n, 4), np.float32)
    pos[:, :3] = rng.uniform(-0.97, 0.97, (n, 3))
    vel = np.zeros((n, 4), np.float32)
    vel[:, :3] = rng.uniform(-0.01, 0.01, (n, 3))
    P = make_params(n, 64, 1.0 / 64.0)
    OP = orc.params_from(P)
    ps = ParticleSystem(n, (64,) * 3, context=gpu_ctx)
    ps.m_params = P
    ps.setArray(ps.POSITION, pos, 0, n)
    ps.setArray(ps.VELOCITY, vel, 0, n)
    st = orc.State(pos, vel, P.numCells)
    print(n, flush=True)
    ps.run(0.5, 4)
    ps.update(0.5)
    for _ in range(5):
        st.update(0.5, OP)
    _compare_system(ps, st)
    ps.close()
    # the reference's stages on caller-owned arrays
    h, i = orc.sort_pairs(*orc.calc_hash(pos, OP))
    cs, ce, sp, sv = orc.reorder(h, i, pos, vel, P.numCells)
    nv = Stages(gpu_ctx, P).collide(sp, sv, i, cs, ce, vel)
    onv = orc.collide(sp, sv, i, cs, ce, OP, newVel4=vel)
    assert np.array_equal(bits(nv), bits(onv))


def test_flat_grid_at_the_walls(gpu_ctx, many):
    walls.test_system_at_the_walls(gpu_ctx, (32, 4, 8))


@pytest.mark.parametrize("pile", [2, 63, 64, 200])
def test_moving_piles_of_other_sizes(gpu_ctx, many, pile):
    walls.test_piles_that_move_as_a_whole(gpu_ctx, pile)

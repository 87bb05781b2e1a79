"""The collide's neighbour walk where cell indices wrap, and its overflowing
lists, against the oracle bit for bit (20,000 spheres: with one radius the
row-split kernel, with radii of their own the row-range one;
test_gpu_row_range.py repeats the former at 40,000).

 - A grid that covers the box exactly: every wall sphere has neighbour cells
   on the opposite side, which the walls put out of contact.
 - The same cells on caller-owned arrays, with spheres outside the grid that
   touch others through the wrap (they must be found), and without.
 - Radii from pos.w: each sphere's own candidate bound, piles of hundreds.
"""
from __future__ import annotations

import os

import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_parity import Stages, _compare_system, bits

pytestmark = pytest.mark.gpu

N, GRID, R = 20000, 32, 1.0 / 32.0


@pytest.fixture(scope="module", autouse=True)
def _oracle_threads():
    orc.set_threads(max(1, min(16, os.cpu_count() or 1)))
    yield
    orc.set_threads(1)


def state(seed, lo=-0.97, hi=0.97, shell=0.5):
    """Random spheres, a share of them near the walls; vel U(+-0.01)."""
    rng = np.random.default_rng(seed)
    pos = np.ones((N, 4), np.float32)
    pos[:, :3] = rng.uniform(lo, hi, (N, 3))
    k = int(N * shell)
    axis = rng.integers(0, 3, k)
    pos[np.arange(k), axis] = np.where(rng.random(k) < 0.5, lo, hi) + rng.uniform(-0.01, 0.01, k)
    vel = np.zeros((N, 4), np.float32)
    vel[:, :3] = rng.uniform(-0.01, 0.01, (N, 3))
    return pos, vel


# gridSize 32 covers the box exactly, 64 with room, 16 not at all (positions
# beyond the grid: every wrap has to be walked)
@pytest.mark.parametrize("grid", [(32, 32, 32), (64, 32, 64), (16, 16, 16), (32, 4, 8)])
def test_system_at_the_walls(gpu_ctx, grid):
    from fullc0ntact_amd import ParticleSystem, make_params
    pos, vel = state(1)
    ps = ParticleSystem(N, grid, context=gpu_ctx)
    ps.m_params = make_params(N, GRID, R, gridSize=grid, numCells=int(np.prod(grid)))
    ps.setArray(ps.POSITION, pos, 0, N)
    ps.setArray(ps.VELOCITY, vel, 0, N)
    st = orc.State(pos, vel, ps.m_params.numCells)
    P = orc.params_from(ps.m_params)
    print(grid, flush=True)
    ps.update(0.5)
    ps.run(0.5, 5)
    for _ in range(6):
        st.update(0.5, P)
    _compare_system(ps, st)
    ps.close()


@pytest.mark.parametrize("outside", [False, True])
def test_stages_through_the_wrap(gpu_ctx, outside):
    from fullc0ntact_amd import make_params
    P = make_params(N, GRID, R)
    OP = orc.params_from(P)
    S = Stages(gpu_ctx, P)
    for call in range(3):
        pos, vel = state(20 + call, -0.99, 0.99)
        if outside and call != 1:  # a call with none in between
            # beyond a wall, hashed to the other side, touching the wall's own
            pos[::40, call % 3] = np.float32(-1.004)
            pos[1::40] = pos[::40]
            pos[1::40, call % 3] = np.float32(-0.98)
        print(outside, call, flush=True)
        h, i = orc.sort_pairs(*orc.calc_hash(pos, OP))
        cs, ce, sp, sv = orc.reorder(h, i, pos, vel, P.numCells)
        nv = S.collide(sp, sv, i, cs, ce, vel)
        onv = orc.collide(sp, sv, i, cs, ce, OP, newVel4=vel)
        assert np.array_equal(bits(nv), bits(onv))
        if outside and call != 1:
            assert np.any(nv[::40] != vel[::40])


@pytest.mark.parametrize("pile", [0, 60, 300])
def test_own_radii_and_piles(gpu_ctx, pile):
    from fullc0ntact_amd import ParticleSystem, make_params
    rng = np.random.default_rng(pile)
    pos, vel = state(3)
    pos[:, 3] = R * np.clip(0.577 * np.exp(0.25 * rng.standard_normal(N)), 1.0 / 3.0, 1.0)
    for c in range(10 if pile else 0):  # piles in cells and across their edges
        k = slice(c * pile, (c + 1) * pile)
        pos[k, :3] = rng.uniform(-0.8, 0.8, 3) + rng.normal(0.0, 0.4 * R, (pile, 3))
    perm = rng.permutation(N)
    pos, vel = pos[perm], vel[perm]
    ps = ParticleSystem(N, (GRID,) * 3, context=gpu_ctx)
    ps.m_params = make_params(N, GRID, R)
    ps.setArray(ps.POSITION, pos, 0, N)
    ps.setArray(ps.VELOCITY, vel, 0, N)
    ps.setPolydisperse(True)
    st = orc.State(pos, vel, ps.m_params.numCells)
    P = orc.params_from(ps.m_params)
    print(pile, flush=True)
    ps.update(0.5)
    ps.run(0.5, 4)
    for _ in range(5):
        orc.update_ex(st, 0.5, P, None, poly=True)
    _compare_system(ps, st)
    ps.close()


@pytest.mark.parametrize("pile", [2, 63, 64, 65, 200, 700])
def test_piles_that_move_as_a_whole(gpu_ctx, pile):
    """Cells all of whose spheres leave in one step, beginning anywhere in a
    64-sphere tile and going on past it: their table entries are cleared (in a
    run, by the changer pass).  No pair forces, a cell's edge per step."""
    from fullc0ntact_amd import ParticleSystem, make_params
    pos, vel = state(4)
    rng = np.random.default_rng(pile)
    edge = 2.0 / GRID
    for c in range(12):
        k = slice(c * pile, (c + 1) * pile)
        cell = rng.integers(4, GRID - 12, 3)
        pos[k, :3] = -1.0 + edge * (cell + 0.5) + rng.uniform(-0.2, 0.2, (pile, 3)) * edge
        vel[k, :3] = edge / 0.5 * np.array([(c % 3 == a) for a in range(3)], np.float32)
    if pile > 64:  # one of a pile stays behind
        vel[11 * pile, :3] = 0.0
    ps = ParticleSystem(N, (GRID,) * 3, context=gpu_ctx)
    ps.m_params = make_params(N, GRID, R, spring=0.0, damping=0.0, shear=0.0)
    ps.setArray(ps.POSITION, pos, 0, N)
    ps.setArray(ps.VELOCITY, vel, 0, N)
    st = orc.State(pos, vel, ps.m_params.numCells)
    P = orc.params_from(ps.m_params)
    print(pile, flush=True)
    ps.run(0.5, 5)
    for _ in range(5):
        st.update(0.5, P)
    _compare_system(ps, st)
    ps.close()

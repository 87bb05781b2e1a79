"""Runs of a system (captured steps) before and after a mesh call on the same
context that needs more sort scratch than the system, against the oracle bit
for bit."""
from __future__ import annotations

import numpy as np
import pytest

from fullc0ntact_amd import meshes
from oracle import oracle as orc
from test_gpu_parity import _compare_system

pytestmark = pytest.mark.gpu


# up to 4,096 spheres and, on a grid of too many rows, the radix sort
@pytest.mark.parametrize("n,grid", [(4096, (64, 64, 64)), (8000, (4, 1024, 512))])
@pytest.mark.parametrize("call", ["labels", "map", "system"])
def test_runs_around_a_call(n, grid, call):
    from fullc0ntact_amd import Context, ParticleSystem, make_params
    from fullc0ntact_amd.distance_map import DistanceMap, mesh_signed_distance
    print(n, grid, call, flush=True)
    rng = np.random.default_rng(n)
    ctx = Context(0)  # of its own: no other test has grown its scratch
    P = make_params(n, grid[0], 1.0 / 64.0, gridSize=grid, numCells=int(np.prod(grid)))
    pos = np.ones((n, 4), np.float32)
    pos[:, :3] = rng.uniform(-0.95, 0.95, (n, 3))
    vel = np.zeros((n, 4), np.float32)
    vel[:, :3] = rng.uniform(-0.01, 0.01, (n, 3))
    ps = ParticleSystem(n, grid, context=ctx)
    ps.m_params = P
    ps.setArray(ps.POSITION, pos, 0, n)
    ps.setArray(ps.VELOCITY, vel, 0, n)
    st = orc.State(pos, vel, P.numCells)
    keep = []
    for part in range(3):
        ps.run(0.5, 12)
        for _ in range(12):
            st.update(0.5, orc.params_from(P))
        _compare_system(ps, st)
        if part == 0:
            v, f = meshes.torus_knot(2, 3, 512, 12, radius=0.12, scale=0.25)
            if call == "labels":
                mesh_signed_distance(ctx, v, f, rng.uniform(-1, 1, (65536, 3)))
            elif call == "map":
                DistanceMap.from_mesh(ctx, v, f, (16,) * 3, 0.125, (-1.0,) * 3).close()
            else:
                keep.append(ParticleSystem(50000, (64,) * 3, context=ctx))
    for s in keep:
        s.close()
    ps.close()
    ctx.close()


def test_open_and_closed_meshes_in_turn():
    """The sorts of an open mesh end at once; those of the meshes and systems
    after it on the same scratch are as ever."""
    from fullc0ntact_amd import Context, ParticleSystem, make_params
    from fullc0ntact_amd.distance_map import mesh_signed_distance
    rng = np.random.default_rng(5)
    ctx = Context(0)
    n, grid = 6000, (4, 1024, 512)  # sorts by radix
    P = make_params(n, grid[0], 1.0 / 64.0, gridSize=grid, numCells=int(np.prod(grid)))
    pos = np.ones((n, 4), np.float32)
    pos[:, :3] = rng.uniform(-0.95, 0.95, (n, 3))
    vel = np.zeros((n, 4), np.float32)
    ps = ParticleSystem(n, grid, context=ctx)
    ps.m_params = P
    ps.setArray(ps.POSITION, pos, 0, n)
    ps.setArray(ps.VELOCITY, vel, 0, n)
    st = orc.State(pos, vel, P.numCells)
    for nu, nv, cut in ((16, 4, 0), (33, 4, 1), (33, 4, 0), (40, 8, 5), (64, 8, 0)):
        v, f = meshes.torus_knot(2, 3, nu, nv, radius=0.2, scale=0.3)
        f = f[:len(f) - cut]
        q = rng.uniform(-1.0, 1.0, (9000, 3))
        print(len(f), cut, flush=True)
        sd, cp = mesh_signed_distance(ctx, v, f, q)
        rsd, rcp, _ = orc.mesh_sdf(v, f, q)
        far = np.abs(rsd) > 1e-14
        assert np.array_equal(sd[far], rsd[far]) and np.array_equal(cp, rcp)
        ps.run(0.5, 11)
        for _ in range(11):
            st.update(0.5, orc.params_from(P))
        _compare_system(ps, st)
    ps.close()
    ctx.close()


def test_map_of_a_mesh_that_is_not_kept(gpu_ctx):
    """A mesh whose copy is too large for the context's scratch (vertices that
    no triangle names) gives the same map."""
    from fullc0ntact_amd.distance_map import DistanceMap
    v, f = meshes.torus_knot(2, 3, 64, 8, radius=0.2, scale=0.3)
    lay = []
    for pad in (0, (256 << 20) // 24):
        w = np.concatenate([v, np.zeros((pad, 3))])
        print(len(w), flush=True)
        m = DistanceMap.from_mesh(gpu_ctx, w, f, (15, 16, 17), 0.125, (-1.0, -1.0, -1.0))
        lay.append(m.download())
        m.close()
    for k in lay[0]:
        assert np.array_equal(lay[0][k], lay[1][k]), k

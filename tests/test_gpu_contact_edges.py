"""Pairs at their contact distance to the last ulp through the row-range
collide: its 16-bit candidate filter (with radii of their own, each sphere's
own bound in binary32), its cell cuts, and those of the launch that takes the
spheres with many candidates, against the oracle bit for bit."""
from __future__ import annotations

import os
import re
from pathlib import Path

import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_parity import _compare_system, _edge_pairs

pytestmark = pytest.mark.gpu

CSRC = Path(__file__).resolve().parents[1] / "fullc0ntact_amd" / "csrc"


@pytest.fixture(scope="module", autouse=True)
def _oracle_threads():
    orc.set_threads(max(1, min(16, os.cpu_count() or 1)))
    yield
    orc.set_threads(1)


def constant(source, name):
    return int(re.search(rf"\b{name} = (\d+)", (CSRC / source).read_text()).group(1))


@pytest.mark.parametrize("poly", [False, True])
def test_edges_through_the_row_range_kernel(gpu_ctx, poly):
    from fullc0ntact_amd import ParticleSystem, make_params
    grid, r = 128, 1.0 / 128.0
    rng = np.random.default_rng(71 + poly)
    pos = _edge_pairs(rng, 9000 if poly else 17000, r, poly)
    if poly:
        # crowds of small spheres around some pairs: more candidates than the
        # row-range kernel takes
        crowd = constant("collide.hpp", "kPileCandidates") + 60
        at = rng.choice(len(pos) // 2, 40, replace=False)
        small = np.zeros((40 * crowd, 4), np.float32)
        small[:, :3] = np.repeat(pos[2 * at, :3], crowd, 0) + rng.uniform(-0.5 * r, 0.5 * r,
                                                                          (40 * crowd, 3))
        small[:, 3] = 0.02 * r
        small[:, :3] = np.clip(small[:, :3], -1.0 + r, 1.0 - r)
        pos = np.concatenate([pos, small])
    n = len(pos)
    assert n > constant("dem_kernels.hip", "kSplitMaxPoly" if poly else "kSplitMaxSpheres")
    pos = pos[rng.permutation(n)]
    vel = np.zeros((n, 4), np.float32)
    # no gravity, no velocities: integrate leaves every position as placed
    P = make_params(n, grid, r, gravity=(0.0, 0.0, 0.0), colliderPos=(50.0, 50.0, 50.0))
    print(poly, n, flush=True)
    for fused in (False, True):
        ps = ParticleSystem(n, (grid,) * 3, context=gpu_ctx)
        ps.m_params = P
        ps.setPolydisperse(poly)
        ps.setArray(ps.POSITION, pos, 0, n)
        ps.setArray(ps.VELOCITY, vel, 0, n)
        st = orc.State(pos, vel, P.numCells)
        for _ in range(3 if fused else 1):
            orc.update_ex(st, 0.5, orc.params_from(P), None, poly=poly)
        if fused:
            ps.run(0.5, 3)
        else:
            ps.update(0.5)
        _compare_system(ps, st)
        if not fused:
            gv = ps.getArray(ps.VELOCITY)
            touched = np.any(gv[:, :3] != 0.0, axis=1)
            assert 0 < touched.sum() < n  # pairs on both sides of the contact distance
        ps.close()

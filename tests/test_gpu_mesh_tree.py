"""The triangle tree of the exact mesh distance against the oracle's brute
force, bit for bit: meshes around its size limits and group remainders,
lattice lines longer than one wave takes, vertices on the surface, meshes that
are not closed (which keep the brute force) and points that are not finite."""
from __future__ import annotations

import os

import numpy as np
import pytest

import distmap_cases as dc
from fullc0ntact_amd import meshes
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _oracle_threads():
    orc.set_threads(max(1, min(16, os.cpu_count() or 1)))
    yield
    orc.set_threads(1)


def box(n):
    """The cube [-1/2, 1/2]^3, 12 n^2 triangles on multiples of 1/n."""
    at, V, F = {}, [], []

    def vid(ax, s, a, b):
        p = [0, 0, 0]
        p[ax], p[(ax + 1) % 3], p[(ax + 2) % 3] = s, a, b
        if tuple(p) not in at:
            at[tuple(p)] = len(V)
            V.append(p)
        return at[tuple(p)]

    for ax in range(3):
        for s in (0, n):
            for i in range(n):
                for j in range(n):
                    a, b = vid(ax, s, i, j), vid(ax, s, i + 1, j)
                    c, d = vid(ax, s, i + 1, j + 1), vid(ax, s, i, j + 1)
                    F += [[a, b, c], [a, c, d]] if s else [[a, c, b], [a, d, c]]
    return np.array(V, np.float64) / n - 0.5, np.array(F, np.uint32)


def mesh(name):
    if name == "open":  # one triangle missing: generalized winding numbers
        v, f = meshes.torus_knot(2, 3, 32, 8, radius=0.2, scale=0.3)
        return v, f[:-1]
    if name == "inverted":
        v, f = box(6)
        return v, f[:, [0, 2, 1]]
    if name == "two":  # overlapping bodies: winding number 2 inside both
        (v, f), (v2, f2) = box(6), box(5)
        return np.concatenate([v, v2 + 0.21]), np.concatenate([f, f2 + len(v)])
    if name.startswith("box"):
        return box(int(name[3:]))
    nu, nv = (int(x) for x in name[4:].split("x"))
    return meshes.torus_knot(2, 3, nu, nv, radius=0.2, scale=0.3)


def check(sd, cp, v, f, q, f32):
    rsd, rcp, _ = orc.mesh_sdf(v, f, q)
    # on the surface (to rounding) the sign is that of a sum near one half
    edge = np.abs(rsd) < 1e-14
    u, t = (np.uint32, np.float32) if f32 else (np.uint64, np.float64)
    a, b = np.ascontiguousarray(sd, t), rsd.astype(t)
    assert np.array_equal(a[~edge].view(u), b[~edge].view(u))
    assert np.array_equal(np.abs(a[edge]).view(u), np.abs(b[edge]).view(u))
    assert np.array_equal(np.ascontiguousarray(cp, t).view(u), rcp.astype(t).view(u))


# 126 and 128 triangles (the tree from 128 on), 3 and 4 levels, a remainder in
# the last group, closed or not, on the lattice's own planes
@pytest.mark.parametrize("name", ["knot9x7", "knot16x4", "knot43x3", "knot171x3", "knot64x32",
                                  "box8", "two", "inverted", "open"])
def test_points(gpu_ctx, name):
    from fullc0ntact_amd.distance_map import mesh_signed_distance
    v, f = mesh(name)
    n = (1 << 24) // len(f) + 65
    print(name, len(f), "triangles", n, "points", flush=True)
    rng = np.random.default_rng(7)
    p = rng.uniform(-1.1, 1.1, (n, 3))
    p[:200] = v[rng.integers(0, len(v), 200)]           # on vertices
    p[200:2000] = np.round(p[200:2000] * 16) / 16       # on the box's planes
    p[2000:2400, 1:] = v[rng.integers(0, len(v), 400), 1:]  # rays through vertices
    sd, cp = mesh_signed_distance(gpu_ctx, v, f, p)
    check(sd, cp, v, f, p, False)


@pytest.mark.parametrize("name,cells", [("box8", (31, 32, 33)), ("knot128x12", (300, 5, 3)),
                                        ("knot64x32", (24, 17, 19)), ("open", (40, 40, 40))])
def test_lattice(gpu_ctx, name, cells):
    from fullc0ntact_amd.distance_map import DistanceMap
    v, f = mesh(name)
    cs = 2.0 / min(cells[0], 32)
    bmin = (-1.0, -1.0, -1.0) if cells[0] < 64 else (-0.5 * cells[0] * cs, -0.15, -0.1)
    print(name, len(f), "triangles", cells, flush=True)
    m = DistanceMap.from_mesh(gpu_ctx, v, f, cells, cs, bmin)
    lay = m.download()
    m.close()
    check(lay["distance"], lay["contact_points"], v, f, dc.lattice_points(cells, cs, bmin), True)


def test_points_not_finite(gpu_ctx):
    from fullc0ntact_amd.distance_map import mesh_signed_distance
    v, f = mesh("knot64x32")
    p = np.random.default_rng(3).uniform(-1, 1, (8192, 3))
    p[5, 0], p[6, 1], p[7], p[8] = np.nan, np.inf, 1e200, 1e20
    sd, cp = mesh_signed_distance(gpu_ctx, v, f, p)
    rsd, rcp, _ = orc.mesh_sdf(v, f, p)
    assert np.array_equal(sd, rsd) and np.array_equal(cp, rcp)


@pytest.mark.parametrize("name", ["knot512x16", "knot513x16"])
def test_points_of_either_key(gpu_ctx, name):
    """The largest mesh whose triangles are ordered by the short key (16,384)
    and the next."""
    from fullc0ntact_amd.distance_map import mesh_signed_distance
    v, f = mesh(name)
    q = np.random.default_rng(11).uniform(-0.8, 0.8, (300, 3))
    q[:20] = v[:20]
    print(name, len(f), flush=True)
    sd, cp = mesh_signed_distance(gpu_ctx, v, f, q)
    check(sd, cp, v, f, q, False)

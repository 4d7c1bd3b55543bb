"""bmf_stitch (seams between the chunks of a world octree) on the GPU against
the oracle's point-by-point formulation, which the CPU tests check against
the restated WorldStitcher recursion.

Bar: the triangle soup bit-exact with the oracle, in the same order, on
worlds of one to three levels of detail and on the terrain of the uneven-LOD
workload at full scale; the GPU's chunk meshes (extracted on the node
lattice) and its seams close a sphere; capacity and argument errors.
"""
from collections import Counter

import numpy as np
import pytest

from binarymeshfitting_amd import capi, workloads as wl

pytestmark = pytest.mark.gpu

WORLDS = [  # (world size, build focus, max level, chunk resolution)
    (32.0, (5.0, 3.0, 2.0), 2, 8),
    (64.0, (10.0, 0.0, 0.0), 3, 8),
    (40.0, (30.0, 3.0, -20.0), 3, 16),
]


@pytest.fixture(scope="module")
def ctx():
    with capi.Context(max_chunks=1024, max_samples=200 * 33 ** 3, max_vertices=1 << 21, max_indices=1 << 23) as c:
        yield c


def _world(W, focus, maxl):
    return wl.lod_world(world_size=W, build_focus=focus, params=wl.LodParams(max_level=maxl, min_level=1))


@pytest.mark.parametrize("world", WORLDS, ids=["uniform", "two-lod", "three-lod"])
@pytest.mark.parametrize("sampler", ["sphere", "terrain", "noise2d", "noise3d"])
def test_stitch_matches_oracle(ctx, oracle, world, sampler):
    W, focus, maxl, dim = world
    nodes, leaves = _world(W, focus, maxl)
    if sampler == "sphere":
        sd = dict(kind=capi.SAMPLER_SPHERE, world_size=2 * W)
    elif sampler == "terrain":
        sd = {**wl.terrain_sampler(), "y0": 0.0, "amp": W / 4, "freq": 0.05}
    elif sampler == "noise2d":  # the reference world's sampler, scaled to the small worlds
        sd = {**capi.noise_preset(capi.PRESET_WORLD), "g_scale": 2.0, "height": W / 4}
    else:
        sd = {**capi.noise_preset(capi.PRESET_TERRAIN3D_PERT), "g_scale": 1.0, "height": W / 4}
    ctx.set_sampler(**sd)
    rc, tris, n = ctx.stitch(nodes, leaves, dim)
    capi.check(rc, "bmf_stitch")
    ref = oracle.stitch_points(oracle.SamplerSpec(**sd), nodes, leaves, dim)
    print(f"{sampler}: {len(leaves)} chunks, {n} seam triangles")
    assert n == len(ref) and n > 0
    assert np.array_equal(tris, ref)


def test_stitch_terrain_world_at_scale(ctx, oracle):
    """The uneven-LOD workload's terrain (7 octaves, frequency 0.005) over a
    4096-unit world split around a focus on the surface, 33^3... here 32^3
    unit nodes per chunk."""
    p = wl.LodParams(max_level=7, min_level=1)
    nodes, leaves = wl.lod_world(world_size=4096.0, build_focus=(300.0, 32.0, -200.0), params=p)
    sd = wl.terrain_sampler(wl.TerrainParams(octaves=7, freq=0.005))
    ctx.set_sampler(**sd)
    rc, tris, n = ctx.stitch(nodes, leaves, 32, cap_triangles=1 << 21)
    capi.check(rc, "bmf_stitch")
    ref = oracle.stitch_points(oracle.SamplerSpec(**sd), nodes, leaves, 32, cap=1 << 21)
    print(f"{len(nodes)} nodes, {len(leaves)} chunks, {n} seam triangles")
    assert n == len(ref) and n > 0
    assert np.array_equal(tris, ref)


def test_gpu_chunks_and_seams_close_a_sphere(ctx):
    W, focus, maxl, dim = WORLDS[2]
    nodes, leaves = _world(W, focus, maxl)
    ctx.set_sampler(kind=capi.SAMPLER_SPHERE, world_size=2 * W)
    rc, seams, n = ctx.stitch(nodes, leaves, dim)
    capi.check(rc, "bmf_stitch")
    cd = [capi.chunk_desc(tuple(float(v) for v in nodes[L]["pos"]),
                          float(np.float32(nodes[L]["size"]) * np.float32(dim - 1) / np.float32(dim)), dim, 0.0, 0, 0)
          for L in leaves]
    ctx.extract(cd, capi.MODE_BATCHED)
    rc, res, _, _ = ctx.results(len(cd))
    capi.check(rc, "bmf_result")
    tris = [seams]
    for j, r in enumerate(res):
        if r.vertex_count:
            pos, idx, _ = ctx.mesh(j)
            p = pos * np.float32(r.delta) + np.asarray(tuple(r.overlap_pos), np.float32)
            tris.append(p[idx.reshape(-1, 3)])
    T = np.concatenate(tris)
    _, inv = np.unique(np.round(T.reshape(-1, 3) / 1e-3).astype(np.int64), axis=0, return_inverse=True)
    F = inv.reshape(-1, 3)
    F = F[(F[:, 0] != F[:, 1]) & (F[:, 1] != F[:, 2]) & (F[:, 0] != F[:, 2])]
    edges = Counter()
    for a, b, c in F:
        for u, v in ((a, b), (b, c), (c, a)):
            edges[(min(u, v), max(u, v))] += 1
    assert set(Counter(edges.values())) == {2}
    assert len(np.unique(F)) - len(edges) + len(F) == 2


def test_stitch_errors(ctx):
    W, focus, maxl, dim = WORLDS[0]
    nodes, leaves = _world(W, focus, maxl)
    ctx.set_sampler(kind=capi.SAMPLER_SPHERE, world_size=2 * W)
    rc, _, n = ctx.stitch(nodes, leaves, dim)
    capi.check(rc, "bmf_stitch")
    rc, _, need = ctx.stitch(nodes, leaves, dim, cap_triangles=n - 1)
    assert rc == capi.ECAPACITY and need == n
    rc, _, _ = ctx.stitch(nodes, leaves, 12)  # not a power of two
    assert rc == capi.EINVAL


@pytest.mark.parametrize("dim", [128, 256])
def test_stitch_deep_worlds(ctx, oracle, dim):
    """A world of 21 levels (the most a morton code holds): with 128 unit
    nodes per chunk edge the last size of the 32-bit lattice coordinates,
    with 256 the first of the 64-bit ones; a few of its chunks, bit-exact
    with the oracle."""
    nodes, leaves = _world(64.0, (0.01, 0.0, 0.0), 21)
    assert int(nodes["level"].max()) == 21
    level, ground = nodes["level"][leaves], nodes["pos"][leaves][:, 1] == 0.0
    leaves = np.concatenate([leaves[(level == 2) & ground][:1], leaves[level == 21][:1]]).astype(np.int32)
    sd = {**wl.terrain_sampler(), "y0": 0.0, "amp": 8.0, "freq": 0.05}
    ctx.set_sampler(**sd)
    rc, tris, n = ctx.stitch(nodes, leaves, dim, cap_triangles=1 << 18)
    capi.check(rc, "bmf_stitch")
    ref = oracle.stitch_points(oracle.SamplerSpec(**sd), nodes, leaves, dim, cap=1 << 18)
    assert n == len(ref) and n > 0
    assert np.array_equal(tris, ref)


def test_stitch_leaf_lists_off_the_tree(ctx, oracle):
    """Leaf list entries that a descent does not end in (an inner node, an
    index out of range, a leaf given twice) keep their meaning."""
    W, focus, maxl, dim = WORLDS[1]
    nodes, leaves = _world(W, focus, maxl)
    inner = int(np.flatnonzero(nodes["world_leaf"] == 0)[-1])
    odd = np.concatenate([leaves[:5], [inner, leaves[2], len(nodes) + 3, -1], leaves[5:]]).astype(np.int32)
    ctx.set_sampler(kind=capi.SAMPLER_SPHERE, world_size=2 * W)
    rc, tris, n = ctx.stitch(nodes, odd, dim)
    capi.check(rc, "bmf_stitch")
    rc, plain, n0 = ctx.stitch(nodes, leaves, dim)
    capi.check(rc, "bmf_stitch")
    rc, twice, n2 = ctx.stitch(nodes, np.array([leaves[2]], np.int32), dim)
    capi.check(rc, "bmf_stitch")
    assert n == n0 + n2
    rows = lambda a: sorted(map(tuple, a.reshape(len(a), 9).tolist()))  # noqa: E731
    assert rows(tris) == rows(np.concatenate([plain, twice]))

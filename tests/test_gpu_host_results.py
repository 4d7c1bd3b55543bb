"""Results, counters and formatted totals that the kernels write to the host:
batches around the wave and segment edges of the format plan's prefix, frames
enqueued back to back, single chunks whose descriptor goes with the launch,
an overflow and an empty batch.  Exact comparisons with the arrays in device
memory and with the other mode."""
import ctypes as C

import numpy as np
import pytest

from binarymeshfitting_amd import capi, workloads

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with capi.Context(max_chunks=2200, max_samples=2200 * 64, max_vertices=1 << 18, max_indices=1 << 20) as c:
        c.set_sampler(**workloads.terrain_sampler())
        yield c


def _chunks(n, seed):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(n):  # around the ground, so with and without a mesh
        dim = int(rng.integers(2, 5))
        out.append(workloads.Chunk(tuple(rng.uniform((0, 20, 0), (200, 44, 200))), 4.0 * (dim - 1), dim, 0.0, 1, 0))
    return out


def _device(ctx, n):
    rc, res, nv, ni = ctx.results(n)
    capi.check(rc, "bmf_result")
    view = capi.MeshView()
    capi.check(capi.lib().bmf_mesh_view_get(ctx.h, C.byref(view)), "bmf_mesh_view_get")
    pos = capi.device_to_numpy(view.positions, (view.total_vertices, 3), np.float32)
    idx = capi.device_to_numpy(view.indices, (view.total_indices,), np.uint32)
    assert nv == view.total_vertices == sum(r.vertex_count for r in res)
    assert ni == view.total_indices == sum(r.index_count for r in res)
    return [(pos[r.vertex_offset:r.vertex_offset + r.vertex_count], idx[r.index_offset:r.index_offset + r.index_count])
            for r in res]


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, 2100])
def test_format_takes_the_chunks_in_order(ctx, n):
    ctx.extract(workloads.to_capi(_chunks(n, n)), capi.MODE_BATCHED)
    meshes = [m for m in _device(ctx, n) if len(m[0])]
    rc, V, I, pos, _, _, idx = ctx.format(space=capi.SPACE_GRID, colors=capi.COLOR_NONE, global_indices=True)
    capi.check(rc, "bmf_format")
    assert V == sum(len(p) for p, _ in meshes) and I == sum(len(i) for _, i in meshes)
    rc, _, _, world, col, _, local = ctx.format(space=capi.SPACE_WORLD, colors=capi.COLOR_WHITE, global_indices=False)
    capi.check(rc, "bmf_format")
    if meshes:
        took = [r for r in ctx.results(n)[1] if r.vertex_count]
        scale = np.repeat(np.array([r.delta for r in took], np.float32), [r.vertex_count for r in took])[:, None]
        shift = np.repeat(np.array([list(r.overlap_pos) for r in took], np.float32), [r.vertex_count for r in took], 0)
        assert np.array_equal(world, pos * scale + shift) and np.all(col == 1.0)
        assert np.array_equal(local, np.concatenate([i for _, i in meshes]))
        first = np.cumsum([0] + [len(p) for p, _ in meshes])
        assert np.array_equal(pos, np.concatenate([p for p, _ in meshes]))
        assert np.array_equal(idx, np.concatenate([i + np.uint32(f) for (_, i), f in zip(meshes, first)]))


def test_modes_agree_and_the_last_frame_counts(ctx):
    frames = [_chunks(40, s) for s in range(6)]
    for f in frames:  # enqueued back to back, none read
        ctx.extract(workloads.to_capi(f), capi.MODE_BATCHED)
    batched = _device(ctx, 40)
    for f in frames:
        ctx.extract(workloads.to_capi(f), capi.MODE_PLAIN)
    plain = _device(ctx, 40)
    assert any(len(p) for p, _ in plain)
    for a, b in zip(batched, plain):
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


def test_overflow_and_empty_batch():
    f = _chunks(60, 3)
    with capi.Context(max_chunks=64, max_samples=64 * 64, max_vertices=40, max_indices=120) as c:
        c.set_sampler(**workloads.terrain_sampler())
        for mode in (capi.MODE_BATCHED, capi.MODE_PLAIN):
            c.extract(workloads.to_capi(f), mode)
            rc, res, nv, ni = c.results(60)
            assert rc == capi.ECAPACITY and nv > 40
            assert sum(r.vertex_count for r in res) <= 40
        c.extract(workloads.to_capi(f[:0]), capi.MODE_BATCHED)
        assert c.results(0)[2] == nv  # an empty batch leaves the counters as they are

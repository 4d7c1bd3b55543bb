"""The word kernels (count, emit, quad vertices and quads) at the edges of
their items: label words that hold many rows or planes (small dims), rows that
end at, before and after a word's last bit, items that end within a plane,
and fields from a single crossing to one at nearly every edge.

External densities, so that the whole mesh is the oracle's bit for bit.
"""
import numpy as np
import pytest

from binarymeshfitting_amd import capi, workloads

pytestmark = pytest.mark.gpu

DIMS = [2, 3, 4, 7, 8, 9, 13, 16, 17, 31, 32, 33, 62, 63, 64, 65, 66, 100, 127, 128, 129, 130]
FILLS = ["noise", "sparse", "sheet"]


def _field(dim, fill, seed):
    rng = np.random.default_rng(seed)
    if fill == "noise":  # about half of all edges change sign
        d = rng.standard_normal((dim, dim, dim))
    elif fill == "sparse":  # a few lone samples, corners among them
        d = np.ones((dim, dim, dim))
        at = rng.integers(0, dim, (max(1, dim // 3), 3))
        d[tuple(at.T)] = -0.5
        d[0, 0, 0] = d[-1, -1, -1] = -2.0
    else:
        g = np.arange(dim)
        d = 0.45 * dim + 0.2 * g[:, None, None] - g[None, :, None] + np.sin(0.7 * g)[None, None, :]
    d = d.astype(np.float32)
    d[d == 0.0] = 0.25
    return d


CASES = [(f, q, [d for d in DIMS if f != "noise" or d <= 66]) for f in FILLS for q in (False, True)]
CASES.append(("sheet", False, [255, 256]))  # the widest windows


@pytest.mark.parametrize("fill,quads,dims", CASES,
                         ids=[f"{f}-{'quads' if q else 'triangles'}-{d[-1]}" for f, q, d in CASES])
def test_items_match_oracle(oracle, fill, quads, dims):
    blocks = [_field(d, fill, 100 * d + len(fill)) for d in dims]
    dev = capi.DeviceArray.from_numpy(np.concatenate([b.ravel() for b in blocks]))
    chunks = [workloads.Chunk((0.0, 0.0, 0.0), float(d - 1), d, 0.0, 1, i & 1) for i, d in enumerate(dims)]
    ns = sum(d ** 3 for d in dims)
    room = 3 * ns if fill == "noise" else ns // 4 + 4096
    with capi.Context(max_chunks=len(dims), max_samples=ns, max_vertices=room, max_indices=6 * room) as ctx:
        ctx.set_sampler(kind=capi.SAMPLER_EXTERNAL, densities=dev)
        if quads:
            ctx.set_mesh_options(mesh=capi.MESH_QUADS)
        ctx.extract(workloads.to_capi(chunks), capi.MODE_BATCHED)
        rc, res, _, _ = ctx.results(len(chunks))
        capi.check(rc, "bmf_result")
        for j, (c, dens) in enumerate(zip(chunks, blocks)):
            if quads:
                ref = oracle.dmc_mesh(dens)
            else:
                words, _ = oracle.label_grid(dens)
                ref = oracle.mesh_from_masks(dens, oracle.cell_masks(words, c.dim))
            V, nI = len(ref["pos"]), len(ref["idx"])
            assert (res[j].vertex_count, res[j].index_count) == (V, nI), c.dim
            if not V:
                continue
            pos, idx, bnd = ctx.mesh(j)
            assert np.array_equal(idx, ref["idx"]), c.dim
            assert np.array_equal(bnd, ref["boundary"]), c.dim
            if quads:
                want = oracle.smooth_n(ref["pos"], ref["boundary"], ref["idx"], 4, 1, c.boundary_processing)
            else:
                want = oracle.smooth(ref["pos"], ref["boundary"], ref["idx"], 1, c.boundary_processing)
            assert np.array_equal(pos, want), c.dim

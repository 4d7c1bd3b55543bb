"""The word kernels when one workgroup takes all of a batch's items: each wave
stages item after item in the same LDS windows and lists, items of many cells
between items of few or none, so that anything of an item read after the next
one is staged shows.  Meshes are the oracle's bit for bit, both mesh modes.
"""
import numpy as np
import pytest

from binarymeshfitting_amd import capi, workloads

pytestmark = pytest.mark.gpu


def _uneven(dim, seed):
    """Slabs of noise between empty ones."""
    rng = np.random.default_rng(seed)
    d = np.ones((dim, dim, dim), np.float32)
    for x in range(0, dim, 3):
        d[x, :: 1 + x % 4] = rng.standard_normal(d[x, :: 1 + x % 4].shape).astype(np.float32)
    d[d == 0.0] = 0.25
    return d


@pytest.mark.parametrize("quads", [False, True], ids=["triangles", "quads"])
def test_one_workgroup_takes_every_item(oracle, quads):
    dims = [3, 10, 23, 41]
    blocks = [_uneven(d, d) for d in dims]
    dev = capi.DeviceArray.from_numpy(np.concatenate([b.ravel() for b in blocks]))
    chunks = [workloads.Chunk((0.0, 0.0, 0.0), float(d - 1), d, 0.0, 0, 0) for d in dims]
    ns = sum(d ** 3 for d in dims)
    with capi.Context(max_chunks=len(dims), max_samples=ns, max_vertices=3 * ns, max_indices=18 * ns) as ctx:
        ctx.set_sampler(kind=capi.SAMPLER_EXTERNAL, densities=dev)
        if quads:
            ctx.set_mesh_options(mesh=capi.MESH_QUADS)
        ctx.set_tuning(row_blocks=1)
        ctx.extract(workloads.to_capi(chunks), capi.MODE_BATCHED)
        rc, res, _, _ = ctx.results(len(chunks))
        capi.check(rc, "bmf_result")
        for j, (d, dens) in enumerate(zip(dims, blocks)):
            if quads:
                ref = oracle.dmc_mesh(dens)
            else:
                words, _ = oracle.label_grid(dens)
                ref = oracle.mesh_from_masks(dens, oracle.cell_masks(words, d))
            assert (res[j].vertex_count, res[j].index_count) == (len(ref["pos"]), len(ref["idx"])), d
            pos, idx, bnd = ctx.mesh(j)
            assert np.array_equal(idx, ref["idx"]) and np.array_equal(bnd, ref["boundary"]), d
            assert np.array_equal(pos, ref["pos"]), d

"""Many CSG primitives near one item of label words: lists that fill no group of
four, the stage of the vertex placement and the item's ids exactly and by one
more, that fit neither and are read from the chunk's list; batches of few items,
whose samples and cells go to more waves, and of many.  Every sample's value
(full lists) and the meshes are the oracle's bit for bit.
"""
import numpy as np
import pytest

from binarymeshfitting_amd import capi, workloads

pytestmark = pytest.mark.gpu


def _heap(dim, n_spheres, n_boxes):
    """Primitives of a few steps heaped on the chunk's middle, each reaching every item of it that meets the surface."""
    rng = np.random.default_rng(100 * n_spheres + n_boxes)
    c = 0.5 * (dim - 1) + rng.uniform(-0.12, 0.12, (n_spheres + n_boxes, 3)) * dim
    r = rng.uniform(0.15, 0.3, (n_spheres + n_boxes, 3)) * dim
    return dict(kind=capi.SAMPLER_CSG, world_size=256.0,
                spheres=np.concatenate([c[:n_spheres], r[:n_spheres, :1]], 1).astype(np.float32),
                boxes=np.concatenate([c[n_spheres:], r[n_spheres:]], 1).astype(np.float32))


def _compare(oracle, sd, chunks, dim, modes):
    spec = oracle.SamplerSpec(**sd)
    n, ns = len(chunks), dim ** 3
    refs = {}
    for c in {c.pos: c for c in chunks}.values():
        oc = oracle.make_chunk(c.pos, c.size, dim, 0.0, 0, 0)
        delta, opos = oracle.geometry(oc)
        block = oracle.sample_block(spec, dim, opos, delta)
        refs[c.pos] = [oracle.extract_chunk(spec, oc)] + [
            oracle.dmc_mesh(block, spec, opos, delta, placement=p, tol=0.1) for p in (0, 1)] + [block]
    with capi.Context(max_chunks=n, max_samples=n * ns, max_vertices=n * ns // 2, max_indices=3 * n * ns) as ctx:
        ctx.set_sampler(**sd)
        for mode in modes:
            for quads, placement in ((False, 0), (True, capi.PLACE_MASS_POINT), (True, capi.PLACE_QEF)):
                ctx.set_mesh_options(mesh=capi.MESH_QUADS if quads else capi.MESH_TRIANGLES, placement=placement)
                ctx.extract(workloads.to_capi(chunks), mode)
                rc, res, _, _ = ctx.results(n)
                capi.check(rc, "bmf_result")
                for j, c in enumerate(chunks):
                    ref = refs[c.pos][quads + placement if quads else 0]
                    assert len(ref["pos"]) > 0
                    assert (res[j].vertex_count, res[j].index_count) == (len(ref["pos"]), len(ref["idx"])), placement
                    pos, idx, bnd = ctx.mesh(j)
                    assert np.array_equal(idx, ref["idx"]) and np.array_equal(bnd, ref["boundary"]), placement
                    assert np.array_equal(pos, ref["pos"]), placement
        c = chunks[0]
        got = ctx.sample_block(workloads.to_capi([c])[0])
        assert np.array_equal(np.asarray(got).ravel(), np.asarray(refs[c.pos][3]).ravel())


@pytest.mark.parametrize("ns,nb", [(16, 0), (0, 17), (10, 7), (13, 50), (300, 1), (0, 258), (600, 424), (601, 424),
                                   (900, 300)])
def test_one_dense_chunk(oracle, ns, nb):
    dim = 18
    chunk = workloads.Chunk((0.0, 0.0, 0.0), float(dim - 1), dim, 0.0, 0, 0)
    _compare(oracle, _heap(dim, ns, nb), [chunk], dim, (capi.MODE_BATCHED, capi.MODE_PLAIN))


@pytest.mark.parametrize("n", [14, 20], ids=["fewer items than the rules' line", "more"])
def test_batches_of_few_and_many_items(oracle, n):
    dim = 42  # 73 items each
    chunks = [workloads.Chunk((0.5 * (k & 1), 0.0, 0.0), float(dim - 1), dim, 0.0, 0, 0) for k in range(n)]
    _compare(oracle, _heap(dim, 20, 21), chunks, dim, (capi.MODE_BATCHED,))

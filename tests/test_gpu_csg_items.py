"""CSG chunks sampled and placed with each item's own primitives: chunks of few
and ragged items, sample steps from a fraction of a primitive to beyond the
union's floor, coordinates far from the origin, more primitives in an item
than its stage holds, none at all.  Meshes are the oracle's bit for bit.
"""
import numpy as np
import pytest

from binarymeshfitting_amd import capi, workloads

pytestmark = pytest.mark.gpu


def _scene(at, step, n_spheres, n_boxes, seed):
    rng = np.random.default_rng(seed)
    ext = 70.0 * step
    c = rng.uniform(0, ext, (n_spheres + n_boxes, 3)) + np.array([at, 0.5 * at, -at])
    r = rng.uniform(2.0, 9.0, (n_spheres + n_boxes, 3)) * step
    return dict(kind=capi.SAMPLER_CSG, world_size=256.0,
                spheres=np.concatenate([c[:n_spheres], r[:n_spheres, :1]], 1).astype(np.float32),
                boxes=np.concatenate([c[n_spheres:], r[n_spheres:]], 1).astype(np.float32))


@pytest.mark.parametrize("step", [0.25, 1.0, 40.0])
@pytest.mark.parametrize("at", [0.0, 60000.0], ids=["near", "far"])
@pytest.mark.parametrize("ns,nb", [(40, 25), (0, 30), (700, 200), (0, 0)])
def test_meshes_match_oracle(oracle, step, at, ns, nb):
    sd = _scene(at, step, ns, nb, ns + nb)
    spec = oracle.SamplerSpec(**sd)
    chunks = [workloads.Chunk((at + 3.0 * step * k, 0.5 * at, -at + step * k), step * (dim - 1), dim, 0.0, 0, 0)
              for k, dim in enumerate((2, 5, 9, 17, 33, 64, 65))]
    total = sum(c.dim ** 3 for c in chunks)
    with capi.Context(max_chunks=len(chunks), max_samples=total, max_vertices=total, max_indices=6 * total) as ctx:
        ctx.set_sampler(**sd)
        for quads, placement in ((False, 0), (True, capi.PLACE_MASS_POINT), (True, capi.PLACE_QEF)):
            ctx.set_mesh_options(mesh=capi.MESH_QUADS if quads else capi.MESH_TRIANGLES, placement=placement)
            ctx.extract(workloads.to_capi(chunks), capi.MODE_BATCHED)
            rc, res, _, _ = ctx.results(len(chunks))
            capi.check(rc, "bmf_result")
            seen = 0
            for j, c in enumerate(chunks):
                oc = oracle.make_chunk(c.pos, c.size, c.dim, c.overlap, 0, 0)
                if quads:
                    delta, opos = oracle.geometry(oc)
                    ref = oracle.dmc_mesh(oracle.sample_block(spec, c.dim, opos, delta), spec, opos, delta,
                                          placement=placement, tol=0.1)
                else:
                    ref = oracle.extract_chunk(spec, oc)
                assert (res[j].vertex_count, res[j].index_count) == (len(ref["pos"]), len(ref["idx"])), (c, placement)
                seen += res[j].vertex_count
                if res[j].vertex_count:
                    pos, idx, bnd = ctx.mesh(j)
                    assert np.array_equal(idx, ref["idx"]) and np.array_equal(bnd, ref["boundary"]), (c, placement)
                    assert np.array_equal(pos, ref["pos"]), (c, placement)
            assert seen > 0 or ns + nb == 0

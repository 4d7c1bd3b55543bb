"""The terrain's block sampling (signs from noise expansions about block
centres, the rest evaluated) over fields where it may go wrong: chunks of few
and ragged blocks, noise too rough for the expansions, long octave chains,
negative amplitudes and gains, coordinates far from the origin.

Every mesh is the oracle's bit for bit, and so is every label of the full
evaluation.
"""
import numpy as np
import pytest

from binarymeshfitting_amd import capi, workloads

pytestmark = pytest.mark.gpu

CASES = {
    "smooth": dict(freq=0.004, octaves=3),
    "rough": dict(freq=0.35, octaves=4),
    "mixed": dict(freq=0.06, octaves=6),
    "one-octave": dict(freq=0.05, octaves=1),
    "long": dict(freq=0.01, octaves=12),
    "growing": dict(freq=0.02, octaves=5, gain=1.7, lacunarity=1.6),
    "downward": dict(freq=0.02, octaves=5, amp=-24.0),
    "negative-gain": dict(freq=0.03, octaves=4, gain=-0.5),
    "flat": dict(freq=0.02, octaves=5, amp=1e-3),
}


def _chunks(at, spacing):
    out = []
    for k, dim in enumerate((2, 3, 4, 5, 6, 9, 17, 32, 33, 64, 65, 70)):
        ext = spacing * (dim - 1)
        out.append(workloads.Chunk((at + 40.0 * k, 32.0 - 0.5 * ext, -at), ext, dim, 0.0, 0, 0))
    return out


@pytest.mark.parametrize("at,spacing", [(0.0, 1.0), (1000.0, 3.0), (250000.0, 0.5)], ids=["near", "wide", "far"])
@pytest.mark.parametrize("name", list(CASES))
def test_meshes_match_oracle(oracle, name, at, spacing):
    sd = {**workloads.terrain_sampler(), "amp": 24.0 * spacing, **CASES[name]}
    if name == "downward":
        sd["amp"] = -24.0 * spacing
    spec = oracle.SamplerSpec(**sd)
    chunks = _chunks(at, spacing)
    ns = sum(c.dim ** 3 for c in chunks)
    with capi.Context(max_chunks=len(chunks), max_samples=ns, max_vertices=3 * ns, max_indices=16 * ns) as ctx:
        ctx.set_sampler(**sd)
        ctx.extract(workloads.to_capi(chunks), capi.MODE_BATCHED)
        rc, res, _, _ = ctx.results(len(chunks))
        capi.check(rc, "bmf_result")
        total = 0
        for j, c in enumerate(chunks):
            ref = oracle.extract_chunk(spec, oracle.make_chunk(c.pos, c.size, c.dim, c.overlap, c.iters, 0))
            assert (res[j].vertex_count, res[j].index_count) == (len(ref["pos"]), len(ref["idx"])), c
            assert bool(res[j].contains_mesh) == bool(ref["contains_mesh"]), c
            total += res[j].vertex_count
            if res[j].vertex_count:
                pos, idx, bnd = ctx.mesh(j)
                assert np.array_equal(idx, ref["idx"]) and np.array_equal(pos, ref["pos"]), c
                assert np.array_equal(bnd, ref["boundary"]), c
        assert total > 0

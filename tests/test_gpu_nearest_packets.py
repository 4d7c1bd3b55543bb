"""The nearest-target search over packets of neighbouring vertices against the
oracle's exact FP32 search: chunks from the smallest to above the size where
the vertex order takes coarser cells, with packets that are not full; target counts at the edges of a leaf and of a hierarchy level;
targets near, far, clustered, on one line and all in one place.  Every
comparison is exact (lowest index at the minimum FP32 distance)."""
import numpy as np
import pytest

from binarymeshfitting_amd import capi, workloads

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tape():
    with capi.Context(max_chunks=1, max_samples=140 ** 3, max_vertices=1 << 19, max_indices=1 << 21) as c:
        c.set_sampler(**workloads.terrain_sampler())
        with capi.Tape(c, max_dim=140, max_vertices=1 << 18, max_indices=1 << 20, checkpoint_every=4) as t:
            yield t


def _targets(kind, n, pos, rng):
    lo, hi = pos.min(0), pos.max(0)
    if kind == "near":
        t = pos[rng.integers(0, len(pos), n)] + rng.normal(0, 0.3, (n, 3))
    elif kind == "far":
        t = rng.uniform(-1, 1, (n, 3)) * 50 + (hi + 4000)
    elif kind == "clusters":
        t = (lo + (hi - lo) * rng.random((4, 3)))[rng.integers(0, 4, n)] + rng.normal(0, 1e-3, (n, 3))
    elif kind == "line":
        t = lo + (hi - lo) * np.linspace(0, 1, n)[:, None]
    else:  # one place
        t = np.repeat(lo[None] + 1.5, n, 0)
    return np.ascontiguousarray(t[rng.permutation(n)], np.float32)


@pytest.mark.parametrize("dim,iters", [(2, 0), (5, 1), (33, 0), (66, 2), (129, 0), (133, 0)])
@pytest.mark.parametrize("kind,n", [("near", 1), ("near", 64), ("far", 65), ("clusters", 4097), ("line", 127),
                                    ("place", 200), ("near", 30_011)])
def test_packet_search_is_the_exact_search(tape, oracle, dim, iters, kind, n):
    # a chunk that the ground passes through at every size
    size = float(dim - 1)
    info = tape.forward(capi.chunk_desc((3.0, 36.0 - 0.5 * size, -7.0), size, dim, 0.0, iters, 0))
    V = info.vertex_count
    assert V > 0
    pos, _, _ = tape.mesh()
    t = _targets(kind, n, pos.astype(np.float64), np.random.default_rng([dim, n]))
    for _ in range(2):  # again on the same tape: the order's counters are left clear
        _, dldp, near = tape.loss_nearest(capi.DeviceArray.from_numpy(t))
        want, _ = oracle.KDTree(t.astype(np.float64)).nearest_f32(pos, threads=16)
        assert np.array_equal(near, want)
        assert np.array_equal(dldp.numpy()[:V], (pos - t[near]) * (np.float32(2.0) / np.float32(V)))
        assert tape.forward(capi.chunk_desc((3.0, 36.0 - 0.5 * size, -7.0), size, dim, 0.0, iters, 0)).vertex_count == V

"""The work that users of this library have it do, as cases that can be timed.

Every case goes through the C ABI (include/bmf.h) by way of the package's
ctypes binding, on buffers that the caller owns, as an engine's generator
thread or a fitting loop calls it: extract a batch, read the per-chunk
results, format the meshes into vertex buffers; or forward, loss, backward.

    listed()             the cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  the context, descriptors and buffers a program holds
    run(state)           one pass and its outputs
    work(case)           the bytes and operations a pass cannot do without
    exact(case, seed)    the outputs in 64 bits, where the inputs alone define them
"""
import ctypes as C
import functools
import math
import types

import numpy as np
import torch  # before the library: both then share one HIP runtime

from binarymeshfitting_amd import capi, tables, workloads

# Indices per triangle-path vertex on a closed surface is 6; arenas leave room.
_INDEX_ROOM = 7
_RESULT = np.dtype([("vertex_offset", "<i8"), ("index_offset", "<i8"), ("vertex_count", "<i4"),
                    ("index_count", "<i4"), ("contains_mesh", "<i4"), ("status", "<i4"), ("sampled", "<i4"),
                    ("delta", "<f4"), ("overlap_pos", "<f4", 3)], align=True)
assert _RESULT.itemsize == C.sizeof(capi.ChunkResult)
_PRESETS = {"terrain2d": capi.PRESET_TERRAIN2D, "terrain2d_pert": capi.PRESET_TERRAIN2D_PERT,
            "terrain3d": capi.PRESET_TERRAIN3D, "terrain3d_pert": capi.PRESET_TERRAIN3D_PERT,
            "windy3d": capi.PRESET_WINDY3D}
_COLORS = {"none": capi.COLOR_NONE, "white": capi.COLOR_WHITE, "noise": capi.COLOR_NOISE}


def listed():
    return [
        # A player's edit: one 64^3-cell chunk meshed again and read at once, the
        # reference's one-chunk job.  Latency and launches are all of it.
        dict(name="one-chunk", kind="terrain", nx=1, ny=1, nz=1, y=0.0, cells=64, octaves=5, iters=4, overlap=0.0,
             bp=0, plain=True, quads=False, normals=False, as_tris=False, contexts=1, color="white", world=False),
        # Entering a level: the headline batch, 512 chunks of which one layer
        # meets the terrain, meshed, smoothed and formatted for the renderer.
        dict(name="uniform-512", kind="terrain", nx=8, ny=8, nz=8, y=0.0, cells=64, octaves=5, iters=4, overlap=0.0,
             bp=0, plain=False, quads=False, normals=False, as_tris=False, contexts=1, color="white", world=False),
        # Flying over terrain: a stream of such batches alternated over three
        # contexts, each read after the next ones are enqueued.
        dict(name="uniform-stream", kind="terrain", nx=8, ny=8, nz=8, y=0.0, cells=64, octaves=5, iters=4,
             overlap=0.0, bp=0, plain=False, quads=False, normals=False, as_tris=False, contexts=3, color="white",
             world=False),
        # An octree frontier: chunks of three sizes and spacings scattered over a
        # large world, most of them off the surface, 0 to 8 smoothing steps each.
        dict(name="uneven-lod", kind="lod", chunks=1536, world=4096, octaves=7, color="white"),
        # The watcher's step as the focus moves over the default world: the LOD
        # pass fills the queue on the device, its chunks are meshed and coloured.
        dict(name="world-step", kind="world", resolution=32, iters=0, shift=0.1, max_gen=400, color="noise"),
        # A volume with overhangs: perturbed 3D noise, every sample evaluated.
        dict(name="field-3d", kind="field", preset="terrain3d_pert", nx=6, ny=3, nz=6, cells=32, size=64.0, iters=2,
             color="white"),
        # Modelled solids: a CSG union meshed by dual marching cubes with QEF
        # placement (sharp edges), 4^3 chunks of 64^3 cells.
        dict(name="csg-hermite", kind="csg", side=4, cells=64, spheres=200, boxes=100, iters=0, qef=True,
             normals=False, color="none"),
        # Lit terrain from the dual mesh: quads written as triangles, smoothed,
        # with vertex normals and an overlap between neighbours.
        dict(name="quads-lit", kind="terrain", nx=4, ny=2, nz=4, y=0.0, cells=64, octaves=5, iters=4, overlap=0.035,
             bp=1, plain=False, quads=True, normals=True, as_tris=True, contexts=1, color="white", world=True),
        # Fitting a 128^3-cell chunk to a scan of 200,000 points: forward, loss
        # against the fixed target set, gradient of every density.
        dict(name="fit-128", kind="fit", cells=128, iters=8, bp=0, targets=200_000, given=False),
        # Fitting free densities (a grid of parameters) to targets that change
        # with every step, so that the search structure is built each time.
        dict(name="fit-grid", kind="fit", cells=56, iters=4, bp=1, targets=20_000, given=True),
        # Densities from the caller's own sampler, meshed with normals, at a
        # chunk size that fills no word or tile evenly.
        dict(name="given-blocks", kind="given", chunks=48, cells=40, iters=2, bp=1, normals=True, color="white"),
        # Crack-free levels of detail: the seam triangles of a world octree.
        dict(name="seams", kind="seams", resolution=32, world=512, levels=5),
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], its logarithm uniform."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["terrain", "terrain", "terrain", "lod", "world", "field", "csg", "fit", "fit", "given",
                       "seams"])
    if kind == "terrain":
        cells = _log(rng, 12, 140)
        most = max(1, 512 // cells)  # the surface of the listed batch at the most
        contexts = rng.choice([1, 1, 1, 2, 3])
        quads = rng.random() < 0.3
        nx, nz = _log(rng, 1, most), _log(rng, 1, most)
        ny = rng.randint(1, 4)
        plain = nx * ny * nz <= 8 and rng.random() < 0.5
        return dict(kind="terrain", nx=nx, ny=ny, nz=nz, y=32.0 - 0.5 * cells * rng.choice([1, ny]), cells=cells,
                    octaves=rng.randint(3, 7), iters=rng.choice([0, 1, 2, 4, 8]),
                    overlap=rng.choice([0.0, 0.0, 0.035, 0.055]), bp=rng.randint(0, 1), plain=plain, quads=quads,
                    normals=rng.random() < 0.3, as_tris=quads and rng.random() < 0.5, contexts=contexts,
                    color=rng.choice(["none", "white", "white", "noise"]), world=rng.random() < 0.5)
    if kind == "lod":
        return dict(kind="lod", chunks=_log(rng, 48, 1536), world=rng.choice([2048, 4096]), octaves=rng.randint(5, 8),
                    color="white")
    if kind == "world":
        return dict(kind="world", resolution=rng.randint(17, 40), iters=rng.choice([0, 0, 1, 3]),
                    shift=rng.uniform(0.02, 0.5), max_gen=_log(rng, 40, 400), color=rng.choice(["white", "noise"]))
    if kind == "field":
        preset = rng.choice(sorted(_PRESETS))
        return dict(kind="field", preset=preset, nx=rng.randint(1, 6), ny=rng.randint(1, 3), nz=rng.randint(1, 6),
                    cells=rng.randint(15, 33), size=float(rng.choice([32, 64, 96])), iters=rng.randint(0, 4),
                    color="white")
    if kind == "csg":
        return dict(kind="csg", side=rng.randint(1, 4), cells=_log(rng, 20, 64), spheres=_log(rng, 8, 200),
                    boxes=_log(rng, 4, 100), iters=rng.choice([0, 0, 2]), qef=rng.random() < 0.6,
                    normals=rng.random() < 0.3, color="none")
    if kind == "fit":
        return dict(kind="fit", cells=_log(rng, 24, 128), iters=rng.choice([0, 1, 3, 4, 8]), bp=rng.randint(0, 1),
                    targets=_log(rng, 500, 200_000), given=rng.random() < 0.5)
    if kind == "given":
        cells = _log(rng, 12, 100)
        return dict(kind="given", chunks=_log(rng, 1, max(1, 3_000_000 // (cells + 1) ** 3)), cells=cells,
                    iters=rng.choice([0, 1, 2, 4]), bp=rng.randint(0, 1), normals=rng.random() < 0.5, color="white")
    return dict(kind="seams", resolution=rng.choice([8, 16, 32]), world=rng.choice([128, 256, 512]),
                levels=rng.randint(2, 5))


# ---- device buffers and views ----------------------------------------------------------------
class _Raw:
    """Device memory that the library owns, for torch.as_tensor (no copy): good only while its owner lives."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "version": 2,
                                         "strides": None}


def _on_device(a):
    """A numpy array's bytes on the GPU."""
    return torch.from_numpy(np.ascontiguousarray(a).view(np.uint8).reshape(-1).copy()).cuda()


class _State:
    """What a program holds between calls; gives its handles back when dropped."""

    def __init__(self, case):
        self.case = case
        self.ctxs, self.tape = [], None
        self.lib = capi.lib()

    def __del__(self):
        if self.tape is not None:
            self.tape.close()
        for c in self.ctxs:
            c.close()


class _Batch:
    """One batch of chunks with its context and the vertex buffers it is formatted into."""

    def __init__(self, state, sampler, chunks, max_samples, max_vertices, max_chunks=None, options=None,
                 color="white", world=False, plain=False):
        self.n = len(chunks)
        cap_n = max(1, max_chunks or self.n)
        self.ctx = capi.Context(max_chunks=cap_n, max_samples=max(max_samples, 64), max_vertices=max_vertices,
                                max_indices=_INDEX_ROOM * max_vertices)
        state.ctxs.append(self.ctx)
        if options:
            self.ctx.set_mesh_options(**options)
        self.ctx.set_sampler(**sampler)
        self.lib = state.lib
        self.mode = capi.MODE_PLAIN if plain else capi.MODE_BATCHED
        self.descs = capi.chunk_array(workloads.to_capi(chunks)) if chunks else None
        self.res = (capi.ChunkResult * cap_n)()
        self.res_np = np.frombuffer(self.res, _RESULT)
        # the program's vertex buffers, whole in the outputs: zeros past the formatted meshes
        self.pos = torch.zeros((max_vertices, 3), dtype=torch.float32, device="cuda")
        self.idx = torch.zeros((_INDEX_ROOM * max_vertices,), dtype=torch.int32, device="cuda")
        self.col = torch.zeros_like(self.pos) if color != "none" else None
        self.nrm = torch.zeros_like(self.pos) if options and options.get("normals") else None
        self.fmt = capi.FormatOptions(capi.SPACE_WORLD if world else capi.SPACE_GRID, _COLORS[color], int(world))
        self.vbo = capi.Vbo(self.pos.data_ptr(), self.col.data_ptr() if self.col is not None else None,
                            self.nrm.data_ptr() if self.nrm is not None else None, self.idx.data_ptr(), max_vertices,
                            _INDEX_ROOM * max_vertices)
        self.nv, self.ni = C.c_int64(), C.c_int64()

    def extract(self):
        capi.check(self.lib.bmf_extract(self.ctx.h, self.descs, self.n, self.mode), "bmf_extract")

    def read(self, n=None):
        """The per-chunk results, then the meshes as vertex buffers in batch order."""
        n = self.n if n is None else n
        capi.check(self.lib.bmf_result(self.ctx.h, self.res, n, None, None), "bmf_result")
        capi.check(self.lib.bmf_format(self.ctx.h, C.byref(self.fmt), C.byref(self.vbo), C.byref(self.nv),
                                       C.byref(self.ni)), "bmf_format")
        r = self.res_np
        out = {"vertices": r["vertex_count"].copy(), "indices_per_chunk": r["index_count"].copy(),
               "contains": r["contains_mesh"].copy(), "positions": self.pos, "indices": self.idx}
        if self.col is not None:
            out["colors"] = self.col
        if self.nrm is not None:
            out["normals"] = self.nrm
        return out


# ---- inputs ----------------------------------------------------------------------------------
def _terrain(case, seed, amp=24.0, freq=0.02):
    return workloads.terrain_sampler(workloads.TerrainParams(amp=amp, freq=freq, octaves=case["octaves"],
                                                             seed=1337 + seed))


def _meets(chunks, amp=24.0, y0=32.0):
    """The chunks that can meet a terrain of that band: what the sampling arena has to hold."""
    return [c for c in chunks
            if c.pos[1] - c.size * c.overlap - y0 <= amp and c.pos[1] + c.size * (1.0 + c.overlap) - y0 >= -amp]


def _samples(chunks):
    return sum(c.dim ** 3 for c in chunks)


def _blocks(case, seed, n):
    """n blocks of a smooth random field over (cells + 1)^3 samples: a tilted height field with waves."""
    dim = case["cells"] + 1
    g = torch.Generator().manual_seed(1000 + seed)
    out = torch.empty((n, dim, dim, dim), dtype=torch.float32, device="cuda")
    a = torch.arange(dim, dtype=torch.float32, device="cuda")
    for b in range(n):
        r = torch.rand((7, 5), generator=g).tolist()
        d = (0.35 + 0.3 * r[0][0]) * dim - a[None, :, None] + 0.25 * (r[0][1] - 0.5) * a[:, None, None]
        for w in r[1:]:
            k = [2.0 * math.pi * (u - 0.5) / 9.0 for u in w[:3]]
            wave = torch.sin(k[0] * a[:, None, None] + k[1] * a[None, :, None] + k[2] * a[None, None, :]
                             + 6.28 * w[3])
            d = d + (0.02 + 0.05 * w[4]) * dim * wave
        out[b] = d
    return out


def _given_chunks(case, n):
    c = case["cells"]
    return [workloads.Chunk((float(c * b), 0.0, 0.0), float(c), c + 1, 0.0, case["iters"], case["bp"])
            for b in range(n)]


def _given_room(case):
    return 4096 + 10 * case["chunks"] * (case["cells"] + 1) ** 2


def _fit_room(case):
    return 8192 + 12 * (case["cells"] + 1) ** 2


def _targets(case, seed):
    c = case["cells"]
    return workloads.sphere_targets(case["targets"], seed=3 + seed, radius=0.3125 * c, centre=(0.5 * c,) * 3)


@functools.lru_cache(maxsize=8)
def _octree(world, levels, focus):
    p = workloads.LodParams(max_level=levels, min_level=1)
    return workloads.lod_world(world_size=float(world), build_focus=focus, params=p)


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def _prepare_terrain(case, seed):
    s = _State(case)
    c, dim = case["cells"], case["cells"] + 1
    s.batches = []
    for k in range(case["contexts"]):
        chunks = [workloads.Chunk((float(c * (i + k * case["nx"])), case["y"] + c * j, float(c * m)), float(c), dim,
                                  case["overlap"], case["iters"], case["bp"])
                  for i in range(case["nx"]) for j in range(case["ny"]) for m in range(case["nz"])]
        on = _meets(chunks)
        options = dict(mesh=capi.MESH_QUADS if case["quads"] else capi.MESH_TRIANGLES,
                       quads_as_triangles=case["as_tris"], normals=case["normals"])
        s.batches.append(_Batch(s, _terrain(case, seed), chunks, _samples(on), 4096 + 6 * len(on) * dim * dim,
                                options=options, color=case["color"], world=case["world"], plain=case["plain"]))
    return s


def _prepare_lod(case, seed):
    s = _State(case)
    chunks = workloads.mixed_lod(case["chunks"], seed=7 + seed, world=case["world"]).chunks
    on = _meets(chunks)
    room = 65536 + 400 * case["chunks"] * 4096 // case["world"]
    s.batches = [_Batch(s, _terrain(case, seed, freq=0.005), chunks, _samples(on), room, color=case["color"])]
    return s


def _prepare_world(case, seed):
    s = _State(case)
    nodes, leaves = _octree(4096, 7, (0.0, -140.0, 0.0))
    u = workloads.SplitMix64(seed)
    angle = 6.283185307179586 * u.uniform()
    far = 4096.0 * case["shift"]
    p = workloads.LodParams(focus=(far * math.cos(angle), -140.0, far * math.sin(angle)), max_level=7, min_level=1,
                            max_gen=case["max_gen"], chunk_resolution=case["resolution"],
                            process_iters=case["iters"])
    res, cap = case["resolution"], case["max_gen"] + 256
    sampler = capi.noise_preset(capi.PRESET_WORLD, world_size=4096.0, seed=1337 + seed)
    s.batch = _Batch(s, sampler, [], cap * res ** 3, cap * 5 * res * res, max_chunks=cap, color=case["color"],
                     world=True)
    s.params = capi.LodParams.of(p)
    s.nodes, s.list = _on_device(nodes), _on_device(leaves.astype(np.int32))
    s.n_nodes, s.n_list = len(nodes), len(leaves)
    s.flags = torch.zeros(len(nodes), dtype=torch.int32, device="cuda")
    s.dirty = torch.zeros(len(leaves), dtype=torch.int32, device="cuda")
    s.items = torch.zeros((cap, workloads.LOD_ITEM.itemsize // 4), dtype=torch.int32, device="cuda")
    s.cap = cap
    s.nd, s.nc = C.c_int32(), C.c_int32()
    return s


def _prepare_field(case, seed):
    s = _State(case)
    c, size = case["cells"], case["size"]
    n = case["nx"] * case["ny"] * case["nz"]
    chunks = [workloads.Chunk((size * i, size * (j - 0.5 * case["ny"]), size * m), size, c + 1, 0.0, case["iters"], 0)
              for i in range(case["nx"]) for j in range(case["ny"]) for m in range(case["nz"])]
    sampler = capi.noise_preset(_PRESETS[case["preset"]], world_size=256.0, seed=1337 + seed)
    s.batches = [_Batch(s, sampler, chunks, n * (c + 1) ** 3, 4096 + 12 * n * (c + 1) ** 2, color=case["color"])]
    return s


def _prepare_csg(case, seed):
    s = _State(case)
    w = workloads.csg_scene(n_side=case["side"], c=case["cells"], seed=42 + seed, n_spheres=case["spheres"],
                            n_boxes=case["boxes"], iters=case["iters"])
    n, dim = len(w.chunks), case["cells"] + 1
    options = dict(mesh=capi.MESH_QUADS, placement=capi.PLACE_QEF if case["qef"] else capi.PLACE_MASS_POINT,
                   qef_tolerance=0.1, normals=case["normals"])
    s.batches = [_Batch(s, w.sampler, w.chunks, _samples(w.chunks), 4096 + 8 * n * dim * dim, options=options,
                        color=case["color"])]
    return s


def _prepare_given(case, seed):
    s = _State(case)
    n, dim = case["chunks"], case["cells"] + 1
    s.densities = _blocks(case, seed, n)
    torch.cuda.synchronize()  # the library reads them on its own stream
    block = types.SimpleNamespace(ptr=s.densities.data_ptr())
    chunks = _given_chunks(case, n)
    s.batches = [_Batch(s, dict(kind=capi.SAMPLER_EXTERNAL, densities=block), chunks, n * dim ** 3,
                        _given_room(case), options=dict(normals=case["normals"]), color=case["color"])]
    return s


def _prepare_fit(case, seed):
    s = _State(case)
    c, dim = case["cells"], case["cells"] + 1
    room = _fit_room(case)
    ctx = capi.Context(max_chunks=4, max_samples=dim ** 3, max_vertices=room, max_indices=_INDEX_ROOM * room)
    s.ctxs.append(ctx)
    s.densities = None
    if case["given"]:
        s.densities = _blocks(case, seed, 1)[0]
    else:
        # the terrain's surface through the middle of the chunk
        p = workloads.TerrainParams(y0=0.25 * c, seed=1337 + seed)
        ctx.set_sampler(**workloads.terrain_sampler(p))
    s.tape = capi.Tape(ctx, max_dim=dim, max_vertices=room, max_indices=_INDEX_ROOM * room, checkpoint_every=2)
    s.chunk = capi.chunk_desc((0.0, 0.0, 0.0), float(c), dim, 0.0, case["iters"], case["bp"])
    s.targets = torch.from_numpy(_targets(case, seed)).cuda()
    s.near = torch.zeros(room, dtype=torch.int32, device="cuda")
    s.dldp = torch.zeros((room, 3), dtype=torch.float32, device="cuda")
    s.dldd = torch.zeros((dim, dim, dim), dtype=torch.float32, device="cuda")
    # the tape's own mesh lives until its next forward: the program keeps a copy
    s.pos = torch.zeros((room, 3), dtype=torch.float32, device="cuda")
    s.idx = torch.zeros(_INDEX_ROOM * room, dtype=torch.int32, device="cuda")
    s.info, s.loss = capi.TapeInfo(), C.c_float()
    torch.cuda.synchronize()
    if not case["given"]:  # fixed targets: their hierarchy is built once
        capi.check(s.lib.bmf_tape_set_targets(s.tape.h, s.targets.data_ptr(), len(s.targets)), "bmf_tape_set_targets")
    return s


def _prepare_seams(case, seed):
    s = _State(case)
    nodes, leaves = _octree(case["world"], case["levels"], (0.0, 32.0, 0.0))
    ctx = capi.Context(max_chunks=16, max_samples=64, max_vertices=64, max_indices=256)
    s.ctxs.append(ctx)
    ctx.set_sampler(**workloads.terrain_sampler(workloads.TerrainParams(seed=1337 + seed)))
    s.nodes, s.leaves = _on_device(nodes), _on_device(leaves.astype(np.int32))
    s.n_nodes, s.n_leaves = len(nodes), len(leaves)
    s.res = C.c_int32(case["resolution"])
    s.cap = 65536 + 40 * len(leaves) * case["resolution"]
    s.tris = torch.zeros((s.cap, 3, 3), dtype=torch.float32, device="cuda")
    s.nt = C.c_int64()
    return s


# ---- passes ----------------------------------------------------------------------------------
def run(state):
    kind = state.case["kind"]
    if kind == "world":
        return _run_world(state)
    if kind == "fit":
        return _run_fit(state)
    if kind == "seams":
        return _run_seams(state)
    for b in state.batches:
        b.extract()
    got = [b.read() for b in state.batches]
    return got if len(got) > 1 else got[0]


def _run_world(s):
    b = s.batch
    capi.check(s.lib.bmf_lod_queue(b.ctx.h, s.nodes.data_ptr(), s.n_nodes, s.list.data_ptr(), s.n_list,
                                   C.byref(s.params), s.flags.data_ptr(), s.dirty.data_ptr(), s.items.data_ptr(),
                                   s.cap, C.byref(s.nd), C.byref(s.nc)), "bmf_lod_queue")
    capi.check(s.lib.bmf_extract_queued(b.ctx.h, capi.MODE_BATCHED), "bmf_extract_queued")
    out = b.read(s.nc.value)
    out.update(flags=s.flags, dirty=s.dirty, items=s.items)
    return out


def _run_fit(s):
    lib, h = s.lib, s.tape.h
    capi.check(lib.bmf_forward_diff(s.ctxs[0].h, C.byref(s.chunk),
                                    s.densities.data_ptr() if s.densities is not None else None, h),
               "bmf_forward_diff")
    if s.densities is None:
        capi.check(lib.bmf_tape_loss_nearest(h, s.dldp.data_ptr(), s.near.data_ptr(), C.byref(s.loss)),
                   "bmf_tape_loss_nearest")
    else:
        capi.check(lib.bmf_loss_nearest(h, s.targets.data_ptr(), len(s.targets), s.dldp.data_ptr(),
                                        s.near.data_ptr(), C.byref(s.loss)), "bmf_loss_nearest")
    capi.check(lib.bmf_backward_diff(h, s.dldp.data_ptr(), s.dldd.data_ptr()), "bmf_backward_diff")
    capi.check(lib.bmf_tape_get(h, C.byref(s.info)), "bmf_tape_get")
    V, nI = s.info.vertex_count, s.info.index_count
    if V:
        s.pos[:V].copy_(torch.as_tensor(_Raw(s.info.positions, (V, 3), "<f4"), device="cuda"))
    if nI:
        s.idx[:nI].copy_(torch.as_tensor(_Raw(s.info.indices, (nI,), "<i4"), device="cuda"))
    return {"positions": s.pos, "loss": s.loss.value, "dldp": s.dldp, "nearest": s.near, "dldd": s.dldd,
            "indices": s.idx}


def _run_seams(s):
    capi.check(s.lib.bmf_stitch(s.ctxs[0].h, s.nodes.data_ptr(), s.n_nodes, s.leaves.data_ptr(), s.n_leaves,
                                C.byref(s.res), s.tris.data_ptr(), s.cap, C.byref(s.nt)), "bmf_stitch")
    return {"triangles": s.tris, "count": s.nt.value}


# ---- what a pass cannot do without -----------------------------------------------------------
# Operations: the full density (every octave) of about one sample per surface
# vertex (the two ends of its edge, shared with its neighbours), the placement,
# 9 operations per triangle and 9 per ring triangle and step, 3 per vertex and
# step.  Bytes: descriptors in, meshes, colours and normals out; given densities in.
_SIMPLEX = 122  # one noise octave: 117 and 5 around it


def _mesh_work(vertices, per_sample, iters, out_bytes, extra_bytes=0):
    flops = vertices * (per_sample + 15 + 4) + iters * vertices * 39
    return {"bytes": float(extra_bytes + vertices * out_bytes), "flops": float(flops)}


def _out_bytes(case):
    """Bytes per vertex of a formatted mesh: position, six indices, colour, normal."""
    return 12 + 24 + (12 if case.get("color", "none") != "none" else 0) + (12 if case.get("normals") else 0)


def work(case):
    kind, c = case["kind"], case.get("cells", 0)
    if kind == "terrain":
        area = case["contexts"] * case["nx"] * case["nz"] * c * c * (1.0 + 2.0 * case["overlap"]) ** -2
        return _mesh_work(2.7 * area, _SIMPLEX * case["octaves"], case["iters"], _out_bytes(case),
                          case["contexts"] * case["nx"] * case["ny"] * case["nz"] * 32)
    if kind == "lod":
        # about one chunk in fifty of a 4096-unit world meets the surface, mean area 64^2
        met = max(1.0, case["chunks"] * 80.0 / case["world"])
        return _mesh_work(2.0 * met * 3400.0, _SIMPLEX * case["octaves"], 4, _out_bytes(case), case["chunks"] * 32)
    if kind == "world":
        met = 0.4 * case["max_gen"]
        return _mesh_work(2.3 * met * case["resolution"] ** 2, 26 * _SIMPLEX, case["iters"], _out_bytes(case),
                          case["max_gen"] * 56)
    if kind == "field":
        n = case["nx"] * case["ny"] * case["nz"]
        return _mesh_work(1.5 * n * c * c, 9 * _SIMPLEX, case["iters"], _out_bytes(case), n * 32)
    if kind == "csg":
        n = case["side"] ** 3
        return _mesh_work(1.2 * n * c * c, 2 * 24, case["iters"], 12 + 16, n * 32)
    if kind == "given":
        n = case["chunks"]
        return _mesh_work(2.5 * n * c * c, 0, case["iters"], _out_bytes(case), n * 4 * (c + 1) ** 3)
    if kind == "fit":
        V, n3 = 2.7 * c * c, (c + 1) ** 3
        w = _mesh_work(V, 0 if case["given"] else 5 * _SIMPLEX, 2 * case["iters"], 12 + 24 + 12 + 4,
                       4 * n3 * (2 if case["given"] else 1) + 12 * case["targets"])
        w["flops"] += V * 8 * math.log2(case["targets"])  # a descent to one target
        return w
    leaves = len(_octree(case["world"], case["levels"], (0.0, 32.0, 0.0))[1])
    tris = 4.0 * leaves ** 0.5 * case["resolution"] * 8
    return {"bytes": 72.0 * 1.2 * leaves + 36.0 * tris, "flops": tris * 2 * 5 * _SIMPLEX}


# ---- 64 bits ---------------------------------------------------------------------------------
# Given densities define the whole result: labels are their signs, and vertex
# placement, smoothing, loss and gradient follow from them.  The samplers' noise
# is this library's own definition (its lattice hash), so that nothing outside of
# it says what their meshes are.
def _mesh64(d, iters, bp):
    """Positions [V][3] and triangles [T][3] of one block, differentiable in d."""
    n = d.shape[0]
    lab = d < 0
    flags = torch.zeros((n, n, n, 3), dtype=torch.bool, device=d.device)
    flags[:-1, :, :, 0] = lab[:-1] ^ lab[1:]
    flags[:, :-1, :, 1] = lab[:, :-1] ^ lab[:, 1:]
    flags[:, :, :-1, 2] = lab[:, :, :-1] ^ lab[:, :, 1:]
    vid = flags.reshape(-1).cumsum(0).reshape(n, n, n, 3) - 1
    e = flags.nonzero()
    step = torch.nn.functional.one_hot(e[:, 3], 3)
    a, b = e[:, :3], e[:, :3] + step
    s0, s1 = d[a[:, 0], a[:, 1], a[:, 2]], d[b[:, 0], b[:, 1], b[:, 2]]
    pos = a.double() + step.double() * (-s0 / (s1 - s0))[:, None]
    rim = (a == 0).any(1) | (a == n - 1).any(1) | (b == n - 1).any(1)
    mask = torch.zeros((n - 1, n - 1, n - 1), dtype=torch.long, device=d.device)
    for k in range(8):
        x, y, z = k >> 2, (k >> 1) & 1, k & 1
        mask += lab[x:n - 1 + x, y:n - 1 + y, z:n - 1 + z].long() << k
    slots = torch.full((256, 15), -1, dtype=torch.long)
    for m, row in enumerate(tables.TRI_TABLE):
        slots[m, :len(row)] = torch.tensor(row, dtype=torch.long)
    edge = torch.tensor(tables.LOCAL_EDGE, device=d.device)
    cells = ((mask > 0) & (mask < 255)).nonzero()
    local = slots.to(d.device)[mask[cells[:, 0], cells[:, 1], cells[:, 2]]]
    at = edge[local.clamp(min=0)]
    ids = vid[cells[:, None, 0] + at[..., 0], cells[:, None, 1] + at[..., 1], cells[:, None, 2] + at[..., 2],
              at[..., 3]]
    tri = ids[local >= 0].reshape(-1, 3)
    count = torch.zeros(len(pos), dtype=torch.float64, device=d.device)
    count.index_add_(0, tri.reshape(-1), torch.ones(tri.numel(), dtype=torch.float64, device=d.device))
    moved = (count > 0) & (~rim | bool(bp))
    for _ in range(iters):
        centre = pos[tri].mean(1)
        acc = torch.zeros_like(pos).index_add(0, tri.reshape(-1), centre.repeat_interleave(3, 0))
        pos = torch.where(moved[:, None], acc / count.clamp(min=1)[:, None], pos)
    return pos, tri


def _nearest64(p, t):
    best = []
    for part in p.split(2048):
        d2 = ((part[:, None, :] - t[None, :, :]) ** 2).sum(2)
        best.append(d2.argmin(1))
    return torch.cat(best) if best else torch.zeros(0, dtype=torch.long, device=p.device)


def _padded(a, rows):
    """`a` in the program's buffer of that many rows: zeros past it."""
    out = torch.zeros((rows, a.shape[1]), dtype=a.dtype, device=a.device)
    out[:len(a)] = a
    return out


def exact(case, seed):
    if case["kind"] == "given":
        pos = [_mesh64(b.double(), case["iters"], case["bp"])[0] for b in _blocks(case, seed, case["chunks"])]
        pos = _padded(torch.cat(pos), _given_room(case))
        out = {"vertices": None, "indices_per_chunk": None, "contains": None, "positions": pos, "indices": None,
               "colors": None}
        if case["normals"]:
            out["normals"] = None  # their schedule depends on the step count: defined by the library
        return out
    if case["kind"] == "fit" and case["given"]:
        d = _blocks(case, seed, 1)[0].double().requires_grad_(True)
        pos, _ = _mesh64(d, case["iters"], case["bp"])
        t = torch.from_numpy(_targets(case, seed)).cuda().double()
        off = pos - t[_nearest64(pos.detach(), t)]
        loss = (off ** 2).sum() / max(1, len(pos))
        loss.backward()
        room = _fit_room(case)
        return {"positions": _padded(pos.detach(), room), "loss": float(loss),
                "dldp": _padded((2.0 * off / max(1, len(pos))).detach(), room), "nearest": None, "dldd": d.grad, "indices": None}
    return None

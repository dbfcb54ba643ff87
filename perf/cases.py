"""What this framework's speed is measured on: the evaluator's work as a user's
program has it done, through HipEvaluator, HipPatchMap, Batch, Server and the
C ABI entry points of include/osdhip.h.

A case is a dict of plain values; ``kind`` names the path:

* ``refine``  EvalStencils of a uniform refinement table, in place in one
  vertex buffer [control | refined] (what Osd::Mesh::Refine does per frame),
  through a HipStencilTable or, ``raw``, through osdhip_eval_stencils on the
  Far arrays;
* ``limit``   EvalStencils of a limit stencil table with 2 or 5 derivatives;
* ``patches`` EvalPatches at many PatchCoords, in the caller's order or
  through osdhip_eval_patches_sorted;
* ``frame``   one frame of a textured, tessellated surface: patch points,
  tessellation coordinates, P and tangents, normals, face-varying UVs;
* ``pick``    a few surface queries: patch lookup, P with both derivative
  orders, normals;
* ``batch``   many meshes x frames in one graph launch (Batch, autotuned);
* ``serve``   one epoch of the server: admission, frame uploads, evaluation.

Meshes are the cube-spheres with 5 % semi-sharp edges that the tests and
bench.py use.  A topology and its compiled host tables belong to the case;
the control points, primvars and query locations come from the seed.
"""
from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

from opensubdiv_amd import _lib, far, meshes, osd, serve, workloads
from opensubdiv_amd.batch import Batch

D = osd.BufferDescriptor


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # the tutorial's cube (386 refined vertices): nothing but call latency
        dict(name="refine_cube", kind="refine", n=0, level=3, length=3, layout=0, raw=False),
        # a dense character or set piece, refined for display each frame
        dict(name="refine_l3_xyz", kind="refine", n=128, level=3, length=3, layout=0, raw=False),
        # positions and four primvars together, finest level, the table
        # layout that batches and the server use
        dict(name="refine_l4_primvars", kind="refine", n=37, level=4, length=7, layout=2,
             raw=False),
        # a caller that keeps the Far table's arrays itself
        dict(name="refine_l2_raw", kind="refine", n=101, level=2, length=5, layout=0, raw=True),
        # limit positions and tangents at every level-3 vertex of a dense mesh
        dict(name="limit_vertices", kind="limit", n=128, level=3, points=0, outputs=3, length=3,
             layout=0),
        # hair or particle roots: random surface points with curvature
        dict(name="limit_scatter_d2", kind="limit", n=45, level=3, points=150001, outputs=6,
             length=3, layout=0),
        # a dense random sampling of the limit surface, in the caller's order
        dict(name="patches_random", kind="patches", n=128, iso=3, coords=4194304, outputs=3,
             length=3, order="random", sort=False),
        # the same kind of sampling through the entry point made for it
        dict(name="patches_sorted", kind="patches", n=90, iso=3, coords=1500001, outputs=3,
             length=4, order="random", sort=True),
        # one frame of a tessellated, textured, shaded surface
        dict(name="frame_tess", kind="frame", n=40, iso=3, rate=9),
        # a few picks on a small model: lookups, curvature, normals
        dict(name="pick_small", kind="pick", n=16, iso=3, queries=1000),
        # a crowd: uneven meshes with 1..16 frames each in one launch
        dict(name="batch_meshes", kind="batch", meshes=12, mesh_seed=5, n_max=64,
             coords_max=262144, length=7),
        # the server's epoch when a burst of requests has arrived
        dict(name="serve_epoch", kind="serve", topologies=4, mesh_seed=11, n_max=48,
             coords_max=131072, requests=10, length=7),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["refine", "refine", "limit", "patches", "patches", "frame", "pick",
                       "batch", "serve"])
    if kind == "refine":
        level = rng.randint(1, 4)
        n = _log_int(rng, 3, min(128, int(math.sqrt(6.3e6 / 6 / 4 ** level))))
        return dict(kind=kind, n=n, level=level, length=rng.choice([1, 2, 3, 3, 4, 5, 6, 7, 8, 11]),
                    layout=rng.choice([0, 0, 2]), raw=rng.random() < 0.3)
    if kind == "limit":
        outputs = rng.choice([3, 3, 6])
        return dict(kind=kind, n=_log_int(rng, 6, 100), level=rng.randint(2, 3),
                    points=_log_int(rng, 500, 1.5e6 if outputs == 3 else 7e5), outputs=outputs,
                    length=rng.choice([3, 3, 4, 7]), layout=rng.choice([0, 0, 2]))
    if kind == "patches":
        iso = rng.randint(2, 4)
        n = _log_int(rng, 6, 120 if iso < 4 else 40)
        return dict(kind=kind, n=n, iso=iso, coords=_log_int(rng, 500, 4.0e6),
                    outputs=rng.choice([1, 3, 3, 6]), length=rng.choice([1, 2, 3, 3, 4, 7]),
                    order=rng.choice(["random", "patch"]), sort=rng.random() < 0.35)
    if kind == "frame":
        n = _log_int(rng, 6, 64)
        return dict(kind=kind, n=n, iso=rng.randint(2, 3), rate=rng.randint(1, 12))
    if kind == "pick":
        return dict(kind=kind, n=_log_int(rng, 4, 64), iso=rng.randint(2, 4),
                    queries=_log_int(rng, 1, 1e5))
    if kind == "batch":
        return dict(kind=kind, meshes=rng.randint(2, 8), mesh_seed=rng.randint(1, 1 << 20),
                    n_max=rng.randint(10, 32), coords_max=rng.randint(5000, 200000),
                    length=rng.choice([3, 7]))
    return dict(kind=kind, topologies=rng.randint(1, 4), mesh_seed=rng.randint(1, 1 << 20),
                n_max=rng.randint(10, 48), coords_max=rng.randint(5000, 131072),
                requests=rng.randint(1, 10), length=rng.choice([3, 7]))


# ------------------------------------- topologies and their host tables (plans)

@functools.lru_cache(maxsize=8)
def _mesh(n):
    """n = 0: the tutorial's cube; else a cube-sphere, n x n quads a face."""
    if n == 0:
        return meshes.unit_cube(seed=0)
    return meshes.cube_sphere(n, seed=n + 1, radial_noise=0.01, crease_fraction=0.05,
                              sharpness_max=4.0)


@functools.lru_cache(maxsize=4)
def _refine_table(n, level):
    far.set_threads(0)
    t = far.Topology(_mesh(n))
    t.refine_uniform(level)
    return t.stencil_table()


@functools.lru_cache(maxsize=4)
def _patch_table(n, iso, uvs=False):
    far.set_threads(0)
    t = far.Topology(_mesh(n))
    if uvs:
        count, index, _ = meshes.cube_sphere_uvs(n)
        t.set_fvar(count, index)
    p = t.patch_table(iso)
    p.points = p.point_stencils()
    return p


@functools.lru_cache(maxsize=3)
def _limit_table(n, level, points, second):
    far.set_threads(0)
    mesh = _mesh(n)
    if points:
        where = meshes.random_patch_locations(mesh.nfaces, points, seed=n + 7)
    else:
        t = far.Topology(mesh)
        t.refine_uniform(level)
        where = t.vertex_locations(level)
    return _patch_table(n, 3).limit_stencils(*where, second=second)


@functools.lru_cache(maxsize=2)
def _hosts(count, mesh_seed, n_max, coords_max, length):
    specs = workloads.sample_meshes(count, mesh_seed, n_range=(8, n_max), levels=(2, 4),
                                    frames=(1, 16), coords=(max(64, coords_max // 16), coords_max))
    far.set_threads(0)
    return [workloads.compile_mesh(s, length, threads=0) for s in specs]


def _control_points(mesh, length, seed, frames=1):
    """(frames, V, length) float32: deformed positions, then primvars."""
    f = meshes.deform_frames(mesh, frames, seed=seed, extra_primvars=max(0, length - 3))
    return np.ascontiguousarray(f[:, :, :length])


def _spec_mesh(s):
    return meshes.cube_sphere(s.n, seed=s.seed, radial_noise=0.01, crease_fraction=0.05,
                              sharpness_max=4.0)


def _cuda(a):
    a = np.ascontiguousarray(a)
    if a.dtype.fields is not None:
        a = a.view(np.int32)
    return torch.from_numpy(a).to("cuda")


def _locations(case, seed):
    """The seed's random surface locations of a patches or pick case."""
    return meshes.random_patch_locations(_mesh(case["n"]).nfaces,
                                         case.get("coords") or case["queries"], seed=seed + 3)


# ------------------------------------------------------------ prepare and run

def prepare(case, seed):
    return _PREPARE[case["kind"]](case, int(seed))


def run(state):
    return _RUN[state["kind"]](state)


def _prepare_refine(case, seed):
    mesh, t, L = _mesh(case["n"]), _refine_table(case["n"], case["level"]), case["length"]
    nc, nr = mesh.nverts, len(t["sizes"])
    vb = osd.HipVertexBuffer.Create(L, nc + nr)
    vb.UpdateData(_control_points(mesh, L, seed)[0], 0, nc)
    s = dict(kind="refine", vb=vb, src=D(0, L, L), dst=D(nc * L, L, L), n=nr, raw=case["raw"])
    if case["raw"]:
        s["csr"] = [_cuda(t[k]) for k in ("sizes", "offsets", "indices", "weights")]
    else:
        s["table"] = osd.HipStencilTable.Create(t, layout=case["layout"],
                                                keep_csr=case["layout"] == 0)
    return s


def _run_refine(s):
    if s["raw"]:
        p = s["vb"].data.data_ptr()
        _lib.check(_lib.load_hip().osdhip_eval_stencils(
            p, _lib.desc(s["src"]), p, _lib.desc(s["dst"]), *[x.data_ptr() for x in s["csr"]],
            0, s["n"], torch.cuda.current_stream().cuda_stream))
    else:
        assert osd.HipEvaluator.EvalStencils(s["vb"], s["src"], s["vb"], s["dst"], s["table"])
    return s["vb"].data


def _prepare_limit(case, seed):
    t = _limit_table(case["n"], case["level"], case["points"], case["outputs"] == 6)
    L, n = case["length"], len(t["sizes"])
    src = _cuda(_control_points(_mesh(case["n"]), L, seed)[0])
    outs = [torch.empty(n, L, dtype=torch.float32, device="cuda") for _ in range(case["outputs"])]
    return dict(kind="limit", src=src, outs=outs, d=D(0, L, L),
                table=osd.HipStencilTable.Create(t, layout=case["layout"]))


def _run_limit(s):
    args = [a for o in s["outs"] for a in (o, s["d"])]
    assert osd.HipEvaluator.EvalStencils(s["src"], s["d"], *args, s["table"])
    return s["outs"]


def _vertex_points(pt, mesh, L, seed):
    """The vertex buffer [control | patch points] of one frame, filled."""
    nc, npts = mesh.nverts, len(pt.points["sizes"])
    vb = osd.HipVertexBuffer.Create(L, nc + npts)
    vb.UpdateData(_control_points(mesh, L, seed)[0], 0, nc)
    table = osd.HipStencilTable.Create(pt.points)
    assert osd.HipEvaluator.EvalStencils(vb, D(0, L, L), vb, D(nc * L, L, L), table)
    return vb, table


def _prepare_patches(case, seed):
    mesh, pt, L = _mesh(case["n"]), _patch_table(case["n"], case["iso"]), case["length"]
    vb, _ = _vertex_points(pt, mesh, L, seed)
    coords = pt.find(*_locations(case, seed))
    if case["order"] == "patch":
        coords = coords[np.argsort(coords["patchIndex"], kind="stable")]
    n = case["coords"]
    outs = [torch.empty(n, L, dtype=torch.float32, device="cuda") for _ in range(case["outputs"])]
    return dict(kind="patches", vb=vb, coords=_cuda(coords), n=n, outs=outs, d=D(0, L, L),
                patches=osd.HipPatchTable.Create(pt.flat()), sort=case["sort"])


def _run_patches(s):
    t, d = s["patches"], s["d"]
    if not s["sort"]:
        args = [a for o in s["outs"] for a in (o, d)]
        assert osd.HipEvaluator.EvalPatches(s["vb"], d, *args, s["n"], s["coords"], t)
    else:
        cd, none = _lib.desc(d), _lib.Desc(0, 0, 0)
        args = [a for o in s["outs"] for a in (o.data_ptr(), cd)]
        args += [None, none] * (6 - len(s["outs"]))
        _lib.check(_lib.load_hip().osdhip_eval_patches_sorted(
            s["vb"].BindHipBuffer(), cd, *args, s["n"], s["coords"].data_ptr(),
            t.GetPatchArrayBuffer(), t.GetPatchIndexBuffer(), t.GetPatchParamBuffer(),
            torch.cuda.current_stream().cuda_stream))
    return s["outs"]


def _prepare_frame(case, seed):
    mesh, pt = _mesh(case["n"]), _patch_table(case["n"], case["iso"], True)
    vb, table = _vertex_points(pt, mesh, 3, seed)
    _, _, uv = meshes.cube_sphere_uvs(case["n"])
    rng = np.random.default_rng(seed)
    uv = (uv + rng.uniform(-0.2, 0.2, size=uv.shape) / case["n"]).astype(np.float32)
    fs = pt.fvar_stencils()
    uvb = osd.HipVertexBuffer.Create(2, len(uv) + len(fs["sizes"]))
    uvb.UpdateData(uv, 0, len(uv))
    if len(fs["sizes"]):
        assert osd.HipEvaluator.EvalStencils(uvb, D(0, 2, 2), uvb, D(2 * len(uv), 2, 2),
                                             osd.HipStencilTable.Create(fs))
    nf = mesh.nfaces
    rates = (ctypes.c_int * 1)(case["rate"])
    # TESS_QUAD scheme 0: quad faces
    per = _lib.load_hip().osdhip_tess_count(0, 4, 1, ctypes.cast(rates, ctypes.c_void_p))
    n = nf * per
    f32 = dict(dtype=torch.float32, device="cuda")
    return dict(kind="frame", vb=vb, table=table, nc=mesh.nverts, uvb=uvb, rates=rates, nf=nf, n=n,
                map=osd.HipPatchMap(pt.arrays, pt.params),
                patches=osd.HipPatchTable.Create(pt.flat()),
                faces=torch.arange(nf, dtype=torch.int32, device="cuda"),
                sizes=torch.full((nf,), 4, dtype=torch.int32, device="cuda"),
                coords=torch.empty(n, 5, dtype=torch.int32, device="cuda"),
                outs=[torch.empty(n, 3, **f32) for _ in range(4)],
                uvs=torch.empty(n, 2, **f32))


def _run_frame(s):
    E, d = osd.HipEvaluator, D(0, 3, 3)
    vb, n, (P, du, dv, nrm) = s["vb"], s["n"], s["outs"]
    assert E.EvalStencils(vb, d, vb, D(s["nc"] * 3, 3, 3), s["table"])
    _lib.check(_lib.load_hip().osdhip_tess_coords(
        0, 4, 1, ctypes.cast(s["rates"], ctypes.c_void_p), s["nf"], None, s["faces"].data_ptr(),
        s["map"].h, s["sizes"].data_ptr(), s["faces"].data_ptr(), s["nf"],
        s["coords"].data_ptr(), torch.cuda.current_stream().cuda_stream))
    assert E.EvalPatches(vb, d, P, d, du, d, dv, d, n, s["coords"], s["patches"])
    assert osd.limit_normals(du, d, dv, d, nrm, d, n)
    assert E.EvalPatchesFaceVarying(s["uvb"], D(0, 2, 2), s["uvs"], D(0, 2, 2), n, s["coords"],
                                    s["patches"], 0)
    return [P, du, dv, nrm, s["uvs"]]


def _prepare_pick(case, seed):
    mesh, pt = _mesh(case["n"]), _patch_table(case["n"], case["iso"])
    vb, _ = _vertex_points(pt, mesh, 3, seed)
    q = case["queries"]
    return dict(kind="pick", vb=vb, n=q, map=osd.HipPatchMap(pt.arrays, pt.params),
                patches=osd.HipPatchTable.Create(pt.flat()),
                query=[_cuda(a) for a in _locations(case, seed)],
                coords=torch.empty(q, 5, dtype=torch.int32, device="cuda"),
                outs=[torch.empty(q, 3, dtype=torch.float32, device="cuda") for _ in range(7)])


def _run_pick(s):
    d, n, outs = D(0, 3, 3), s["n"], s["outs"]
    assert s["map"].FindPatches(n, *s["query"], s["coords"])
    args = [a for o in outs[:6] for a in (o, d)]
    assert osd.HipEvaluator.EvalPatches(s["vb"], d, *args, n, s["coords"], s["patches"])
    assert osd.limit_normals(outs[1], d, outs[2], d, outs[6], d, n)
    return outs


def _mesh_hosts(case):
    count = case.get("meshes") or case["topologies"]
    return _hosts(count, case["mesh_seed"], case["n_max"], case["coords_max"], case["length"])


def _prepare_batch(case, seed):
    L, dms = case["length"], []
    for h in _mesh_hosts(case):
        d = workloads.DeviceMesh(h)
        F = h.spec.frames
        new = np.zeros((h.nctrl, F, d.lp), np.float32)
        new[:, :, :L] = _control_points(_spec_mesh(h.spec), L, seed + h.spec.index,
                                        F).transpose(1, 0, 2)
        d.vbuf[:new.size].copy_(torch.from_numpy(new.reshape(-1)))
        dms.append(d)
    b = Batch(L, [x for d in dms for x in d.stencil_segments()], [d.patch_segment() for d in dms])
    b.tune(reps=3)                      # the variant its program then keeps
    return dict(kind="batch", batch=b, outs=[[d.refined, *d.out] for d in dms])


def _run_batch(s):
    s["batch"].launch(torch.cuda.current_stream().cuda_stream)
    return s["outs"]


def _requests(case):
    """(topology, kind, frame) of each request of the burst."""
    return [(k * 7 // 2 % case["topologies"], "limit" if k % 2 else "refine", k % 3)
            for k in range(case["requests"])]


def _request_frames(case, h, seed):
    return _control_points(_spec_mesh(h.spec), case["length"], seed + 100 * h.spec.index, 3)


def _prepare_serve(case, seed):
    res = serve.residents_from_hosts(_mesh_hosts(case))
    for r, h in zip(res, _mesh_hosts(case)):
        r.frames = _request_frames(case, h, seed)
    # budgets for two epochs of the largest requests
    most = max(r.nctrl + max(r.nrefine, r.npts + 3 * r.ncoords) for r in res)
    budget = 4 * case["length"] * most * 2 * case["requests"] + (1 << 20)
    sv = serve.Server(res, case["length"], budget, budget, slots=2)
    return dict(kind="serve", server=sv, turn=0, asked=_requests(case))


def _run_serve(s):
    sv, slot = s["server"], s["server"].slots[s["turn"]]
    s["turn"] = (s["turn"] + 1) % len(sv.slots)
    if slot["reqs"] is not None:        # this slot's last epoch: its results are done with
        slot["event"].synchronize()
        for r in slot["reqs"]:
            sv.release(r)
    reqs = [serve.Request(k, t, kind, 0.0, f) for k, (t, kind, f) in enumerate(s["asked"])]
    for r in reqs:
        assert sv.admit(r)
    sv.launch(slot, reqs)
    return [[sv.dev[o:o + m] for o, _, m in sv._pieces(r)] for r in reqs]


_PREPARE = dict(refine=_prepare_refine, limit=_prepare_limit, patches=_prepare_patches,
                frame=_prepare_frame, pick=_prepare_pick, batch=_prepare_batch,
                serve=_prepare_serve)
_RUN = dict(refine=_run_refine, limit=_run_limit, patches=_run_patches, frame=_run_frame,
            pick=_run_pick, batch=_run_batch, serve=_run_serve)


# ------------------------------------------------------- work and tolerances

def _stencil_work(t, nw, L, nc, frames=1):
    """Sizes, indices and weights once; control points read and results
    written once per frame; a multiply and an add per term."""
    n, e = len(t["sizes"]), len(t["indices"])
    return (4 * n + 4 * (1 + nw) * e + 4 * L * frames * (nc + nw * n), 2 * nw * e * L * frames)


def _patch_work(pt, coords, nout, L, npoints, frames=1):
    """Coords, patch tables and points once, results once; 16 points a
    coord, a multiply and an add per term."""
    b = coords * (20 + 4 * L * nout * frames) + 4 * len(pt.indices) + 12 * len(pt.params)
    return b + 4 * L * npoints * frames, 32 * nout * coords * L * frames


def work(case):
    kind, L = case["kind"], case.get("length", 3)
    if kind == "refine":
        b, f = _stencil_work(_refine_table(case["n"], case["level"]), 1, L, _mesh(case["n"]).nverts)
    elif kind == "limit":
        t = _limit_table(case["n"], case["level"], case["points"], case["outputs"] == 6)
        b, f = _stencil_work(t, case["outputs"], L, _mesh(case["n"]).nverts)
    elif kind == "patches":
        pt = _patch_table(case["n"], case["iso"])
        b, f = _patch_work(pt, case["coords"], case["outputs"], L, pt.num_vertices_total)
    elif kind == "frame":
        pt = _patch_table(case["n"], case["iso"], True)
        n = _mesh(case["n"]).nfaces * (case["rate"] + 1) ** 2
        b, f = _stencil_work(pt.points, 1, 3, _mesh(case["n"]).nverts)
        # coords written and read; P, du, dv, normals and UVs written once
        b += n * (2 * 20 + 4 * 14) + 4 * 3 * pt.num_vertices_total + 4 * len(pt.indices) + \
            12 * len(pt.params)
        f += n * (32 * 9 + 20)
    elif kind == "pick":
        pt, n = _patch_table(case["n"], case["iso"]), case["queries"]
        # a few queries touch their own patches' points, not the tables
        b, f = n * (20 + 2 * 20 + 12 + 64 + 16 * 12 + 7 * 12), n * (32 * 18 + 20)
        b = min(b, n * 144 + 12 * pt.num_vertices_total + 4 * len(pt.indices) +
                12 * len(pt.params))
    else:
        b = f = 0
        for k, h in enumerate(_mesh_hosts(case)):
            F, nr, npts, nc = h.spec.frames, int(h.refine.num_stencils), len(h.points["sizes"]), \
                len(h.coords)
            ref = 4 * nr + 8 * int(h.refine.nnz)
            tab = 4 * npts + 8 * len(h.points["indices"]) + 20 * nc + 4 * len(h.indices) + \
                12 * len(h.params)
            frame_ref = 4 * L * (h.nctrl + nr)
            frame_lim = 4 * L * (2 * (h.nctrl + npts) + 3 * nc)
            flop_ref = 2 * L * int(h.refine.nnz)
            flop_lim = L * (2 * len(h.points["indices"]) + 96 * nc)
            if kind == "batch":
                b += ref + tab + F * (frame_ref + frame_lim)
                f += F * (flop_ref + flop_lim)
            else:
                # each request evaluates one frame; a table is read once
                what = [w for topo, w, _ in _requests(case) if topo == k]
                nref, nlim = what.count("refine"), what.count("limit")
                b += ref * (nref > 0) + tab * (nlim > 0) + nref * frame_ref + nlim * frame_lim
                f += nref * flop_ref + nlim * flop_lim
    return {"bytes": int(b), "flops": int(f)}


def tolerance(case):
    """About four times the distance from the same sums in 64 bits (32-bit
    products and sums of 16 to a few dozen terms), measured over the listed
    and drawn cases: positions 1e-7; tangents, whose terms cancel by the
    number of faces around the mesh, up to 7e-6 (n = 128); second
    derivatives up to 7e-5."""
    kind = case["kind"]
    if kind == "refine":
        return {"rel": 3e-7}
    if kind == "limit":
        return {"rel": 8e-6 if case["outputs"] == 3 else 2e-5}
    if kind == "pick" or case.get("outputs") == 6:
        return {"rel": 3e-4}
    if kind == "patches" and case["outputs"] == 1:
        return {"rel": 5e-7}
    if kind in ("patches", "frame"):
        return {"rel": 3e-5}
    return {"rel": 6e-6}


# ---------------------------------------------- the same results in 64 bits

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a, dtype=None):
    x = torch.from_numpy(np.ascontiguousarray(a)).to(_device())
    return x if dtype is None else x.to(dtype)


def _exact_stencils(sizes, indices, weights, src):
    """Rows sum_j w_j src[index_j] of a Far table, src (V, C) float64."""
    n, C = len(sizes), src.shape[1]
    ends = torch.cumsum(_t(sizes, torch.int64), 0)
    begins = ends - _t(sizes, torch.int64)
    idx, w = _t(indices), _t(weights)
    out = torch.zeros(n, C, dtype=torch.float64, device=src.device)
    step = max(1, int(2e8 // (C * max(1, len(indices) // max(1, n)) * 8)))
    for r in range(0, n, step):
        m = min(n, r + step)
        a, b = int(begins[r]), int(ends[m - 1])
        row = torch.repeat_interleave(torch.arange(m - r, device=src.device),
                                      ends[r:m] - begins[r:m])
        out[r:m].index_add_(0, row, src[idx[a:b].long()] * w[a:b].double()[:, None])
    return out


def _bspline(t):
    t2, t3 = t * t, t * t * t
    return ([(1 - t) ** 3 / 6, (3 * t3 - 6 * t2 + 4) / 6, (1 + 3 * t + 3 * t2 - 3 * t3) / 6, t3 / 6],
            [-(1 - t) ** 2 / 2, (3 * t2 - 4 * t) / 2, (1 + 2 * t - 3 * t2) / 2, t2 / 2],
            [1 - t, 3 * t - 2, 1 - 3 * t, t])


def _bernstein(t):
    u = 1 - t
    return ([u ** 3, 3 * u * u * t, 3 * u * t * t, t ** 3],
            [-3 * u * u, 3 * u * u - 6 * u * t, 6 * u * t - 3 * t * t, 3 * t * t],
            [6 * u, 6 * t - 12 * u, 6 * u - 12 * t, 6 * t])


# derivative orders (in s, in t) of P, du, dv, duu, duv, dvv
_ORDERS = [(0, 0), (1, 0), (0, 1), (2, 0), (1, 1), (0, 2)]


def _weights_regular(s, t, boundary, orders):
    cs, ct = _bspline(s), _bspline(t)
    out = []
    for a, b in orders:
        w = [[cs[a][j] * ct[b][i] for j in range(4)] for i in range(4)]
        zero = torch.zeros_like(s)
        # a missing row or column of points is the reflection 2 P1 - P2
        for bit, at in ((1, lambda k, i: (i, k)), (2, lambda k, i: (k, 3 - i)),
                        (4, lambda k, i: (3 - i, k)), (8, lambda k, i: (k, i))):
            on = ((boundary & bit) != 0).to(s.dtype)
            for k in range(4):
                (r0, c0), (r1, c1), (r2, c2) = at(k, 0), at(k, 1), at(k, 2)
                lost = w[r0][c0] * on
                w[r2][c2] = w[r2][c2] - lost
                w[r1][c1] = w[r1][c1] + 2 * lost
                w[r0][c0] = torch.where(on != 0, zero, w[r0][c0])
        out.append(torch.stack([x for row in w for x in row], 1))
    return out


# the Bezier (column, row) of each Gregory point: corner, two edge points and
# two face points at each of the four corners
_GREGORY = [(0, 0), (1, 0), (0, 1), (1, 1), (1, 1), (3, 0), (3, 1), (2, 0), (2, 1), (2, 1),
            (3, 3), (2, 3), (3, 2), (2, 2), (2, 2), (0, 3), (0, 2), (1, 3), (1, 2), (1, 2)]


def _weights_gregory(s, t, orders):
    cs, ct = _bernstein(s), _bernstein(t)
    x, y = 1 - s, 1 - t
    g = [None] * 20
    for c, (num, other) in enumerate(((s, t), (t, x), (x, y), (y, s))):
        den = num + other
        f = torch.where(den > 0, num / torch.where(den > 0, den, torch.ones_like(den)), num)
        g[5 * c + 3], g[5 * c + 4] = f, 1 - f
    return [torch.stack([cs[a][j] * ct[b][i] * (1.0 if g[k] is None else g[k])
                         for k, (j, i) in enumerate(_GREGORY)], 1) for a, b in orders]


def _weights_quad(s, t, orders):
    ls, lt = ([1 - s, s], [-torch.ones_like(s), torch.ones_like(s)]), \
        ([1 - t, t], [-torch.ones_like(t), torch.ones_like(t)])
    zero = torch.zeros_like(s)
    out = []
    for a, b in orders:
        w = [zero if a > 1 or b > 1 else ls[a][j] * lt[b][i]
             for i, j in ((0, 0), (0, 1), (1, 1), (1, 0))]
        out.append(torch.stack(w, 1))
    return out


def _exact_patches(arrays, indices, params, patch, s, t, src, nout):
    """P and the first nout - 1 derivatives at (patch index, ptex s, t) of
    quad patches; src (V, C) float64."""
    dev, orders = src.device, _ORDERS[:nout]
    which = np.repeat(np.arange(len(arrays)), arrays["numPatches"])
    pid = np.arange(len(params))
    base = arrays["indexBase"][which] + arrays["stride"][which].astype(np.int64) * \
        (pid - arrays["primitiveIdBase"][which])
    f1 = params["field1"].astype(np.int64)
    ptype = np.where((f1 >> 5) & 1, arrays["regDesc"][which], arrays["desc"][which])
    base, f1, ptype, idx = _t(base), _t(f1), _t(ptype, torch.int64), _t(indices, torch.int64)
    outs = [torch.zeros(len(patch), src.shape[1], dtype=torch.float64, device=dev)
            for _ in range(nout)]
    chunk = max(1, int(3e8 // (8 * 20 * max(src.shape[1], nout))))
    for c in range(0, len(patch), chunk):
        p = patch[c:c + chunk]
        f = f1[p]
        depth = f & 15
        size = torch.pow(2.0, (depth - ((f >> 4) & 1)).double())
        ss = s[c:c + chunk].double() * size - ((f >> 22) & 1023).double()
        tt = t[c:c + chunk].double() * size - ((f >> 12) & 1023).double()
        scale = torch.pow(2.0, depth.double())
        for kind, npt in ((6, 16), (9, 20), (3, 4)):
            m = torch.nonzero(ptype[p] == kind)[:, 0]
            if not len(m):
                continue
            if kind == 6:
                w = _weights_regular(ss[m], tt[m], (f[m] >> 7) & 31, orders)
            elif kind == 9:
                w = _weights_gregory(ss[m], tt[m], orders)
            else:
                w = _weights_quad(ss[m], tt[m], orders)
            cv = idx[base[p[m]][:, None] + torch.arange(npt, device=dev)].clamp_min(0)
            v = src[cv.reshape(-1)].reshape(len(m), npt, -1)
            for o in range(nout):
                d = (w[o][:, :, None] * v).sum(1) * (scale[m] ** sum(orders[o]))[:, None]
                outs[o][c + m] = d
    return outs


def _exact_find(params, ptex, s, t):
    """The patch that covers each (ptex face, s, t): the deepest cell of its
    face's quadtree, upper halves from their median on."""
    f1 = params["field1"].astype(np.int64)
    face = (params["field0"] & 0xfffffff).astype(np.int64)
    depth = f1 & 15
    key = lambda f, d, u, v: ((f * 16 + d) * 1024 + u) * 1024 + v  # noqa: E731
    have = key(face, depth, (f1 >> 22) & 1023, (f1 >> 12) & 1023)
    order = np.argsort(have)
    have = have[order]
    out = np.full(len(ptex), -1, np.int64)
    for d in range(int(depth.max()) + 1):
        cell = lambda x: np.minimum(np.floor(np.float64(x) * (1 << d)), (1 << d) - 1).astype(np.int64)  # noqa: E731,E501
        k = key(np.asarray(ptex, np.int64), d, cell(s), cell(t))
        at = np.minimum(np.searchsorted(have, k), len(have) - 1)
        out = np.where((have[at] == k) & (out < 0), order[at], out)
    return out


def _exact_points(table, ctrl):
    """[control | patch points] in 64 bits from (V, C) control points."""
    src = _t(ctrl, torch.float64)
    return torch.cat([src, _exact_stencils(table["sizes"], table["indices"], table["weights"],
                                           src)])


def _tess_pattern(rate):
    """Bfr's uniform pattern of a quad: the boundary counter-clockwise from
    (0, 0), then the rings inwards; steps accumulate in 32 bits."""
    f = np.float32
    d = f(1) / f(rate)
    pts = []

    def line(u, v, du, dv, n):
        for _ in range(n):
            pts.append((u, v))
            u, v = f(u + du), f(v + dv)
    one, zero = f(1), f(0)
    line(zero, zero, d, zero, rate)
    line(one, zero, zero, d, rate)
    line(one, one, -d, zero, rate)
    line(zero, one, zero, -d, rate)
    u, left = d, rate - 2
    for _ in range(rate // 2):
        if left > 0:
            far_ = f(one - u)
            line(u, u, d, zero, left)
            line(far_, u, zero, d, left)
            line(far_, far_, -d, zero, left)
            line(u, far_, zero, -d, left)
        else:
            pts.append((f(0.5), f(0.5)))
        u, left = f(u + d), left - 2
    return np.array(pts, np.float32)


def _normals(du, dv):
    n = torch.linalg.cross(du, dv)
    return n / n.norm(dim=1, keepdim=True)


def exact(case, seed):
    kind, seed, L = case["kind"], int(seed), case.get("length", 3)
    if kind == "refine":
        t = _refine_table(case["n"], case["level"])
        return _exact_points(t, _control_points(_mesh(case["n"]), L, seed)[0]).reshape(-1)
    if kind == "limit":
        t = _limit_table(case["n"], case["level"], case["points"], case["outputs"] == 6)
        src = _t(_control_points(_mesh(case["n"]), L, seed)[0], torch.float64)
        return [_exact_stencils(t["sizes"], t["indices"], t[k], src)
                for k in ("weights", "du", "dv", "duu", "duv", "dvv")[:case["outputs"]]]
    if kind in ("patches", "pick"):
        pt, nout = _patch_table(case["n"], case["iso"]), case.get("outputs", 6)
        ptex, s, t = _locations(case, seed)
        src = _exact_points(pt.points, _control_points(_mesh(case["n"]), L, seed)[0])
        patch = _exact_find(pt.params, ptex, s, t)
        s, t = s.astype(np.float32), t.astype(np.float32)
        if case.get("order") == "patch":
            o = np.argsort(patch, kind="stable")
            patch, s, t = patch[o], s[o], t[o]
        outs = _exact_patches(pt.arrays, pt.indices, pt.params, _t(patch), _t(s), _t(t), src, nout)
        return outs + [_normals(outs[1], outs[2])] if kind == "pick" else outs
    if kind == "frame":
        mesh, pt = _mesh(case["n"]), _patch_table(case["n"], case["iso"], True)
        uv = _tess_pattern(case["rate"])
        ptex = np.repeat(np.arange(mesh.nfaces), len(uv))
        s, t = np.tile(uv[:, 0], mesh.nfaces), np.tile(uv[:, 1], mesh.nfaces)
        patch = _t(_exact_find(pt.params, ptex, s, t))
        src = _exact_points(pt.points, _control_points(mesh, 3, seed)[0])
        s, t = _t(s), _t(t)
        outs = _exact_patches(pt.arrays, pt.indices, pt.params, patch, s, t, src, 3)
        base = meshes.cube_sphere_uvs(case["n"])[2]
        rng = np.random.default_rng(seed)
        base = (base + rng.uniform(-0.2, 0.2, size=base.shape) / case["n"]).astype(np.float32)
        fuv = _exact_points(pt.fvar_stencils(), base)
        f = pt.fvar
        uvs = _exact_patches(f["arrays"], f["indices"], f["params"], patch, s, t, fuv, 1)
        return outs + [_normals(outs[1], outs[2])] + uvs
    if kind == "batch":
        return [_exact_mesh(h, _control_points(_spec_mesh(h.spec), L, seed + h.spec.index,
                                               h.spec.frames), True, True)
                for h in _mesh_hosts(case)]
    hosts = _mesh_hosts(case)
    out = []
    for topo, what, frame in _requests(case):
        h = hosts[topo]
        one = _request_frames(case, h, seed)[frame:frame + 1]
        out.append(_exact_mesh(h, one, what == "refine", what == "limit"))
    return out


def _exact_mesh(h, frames, refine, limit):
    """Frame-major refined vertices and / or P, dPdu, dPdv of one mesh."""
    F, nc, L = frames.shape
    src = _t(frames.transpose(1, 0, 2).reshape(nc, F * L), torch.float64)
    major = lambda x: x.reshape(-1, F, L).transpose(0, 1).reshape(-1)  # noqa: E731
    out = []
    if refine:
        r = h.refine
        view = lambda p, t, n: np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(t)), (n,))  # noqa: E731,E501
        n, e = int(r.num_stencils), int(r.nnz)
        out.append(major(_exact_stencils(view(r.sizes_ptr, ctypes.c_int, n),
                                         view(r.indices_ptr, ctypes.c_int, e),
                                         view(r.weights_ptr, ctypes.c_float, e), src)))
    if limit:
        p = h.points
        src = torch.cat([src, _exact_stencils(p["sizes"], p["indices"], p["weights"], src)])
        c = h.coords
        out += [major(x) for x in _exact_patches(h.arrays, h.indices, h.params,
                                                 _t(c["patchIndex"], torch.int64), _t(c["s"]),
                                                 _t(c["t"]), src, 3)]
    return out

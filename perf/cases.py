"""Performance cases of the hot path: what programs built on this library have it do.

Kinds of case (each pass goes through the public entry points):

  step      a lattice edit: the field of one grid (gc.lattice_field) and its indexed mesh
            (gpucad_extract), output buffers preallocated, asynchronous on the stream
  batch     many grids of uneven sizes in one graph replay (gc.Batch)
  serve     a burst of edit requests through the request loop (gc.Server)
  lattice   the reference application's meshing of a synthesised lattice:
            normalise_four, then computeIsosurface_lattice into its own buffers
  boolean   a primitive's field, classify_copy_Voxel, then computeIsosurface
  synth     spatially variant lattice synthesis in one call (gc.svl_field)
  harmonic  the reference's own synthesis loop, harmonic by harmonic
  unit      the unit cell: lattice, transforms, spectrum and its mesh

Sizes come from gpucadforam_amd/configs.py, bench.py and the tests, or lie
between theirs (odd ones among them).
"""
import ctypes as C
import math
import random

import torch

import gpucadforam_amd as gc
from gpucadforam_amd import configs as CF

TPMS = {"gyroid": gc.TPMS_GYROID, "schwarz_p": gc.TPMS_SCHWARZ_P, "diamond": gc.TPMS_DIAMOND}
PRIM = {"none": gc.PRIM_NONE, "sphere": gc.PRIM_SPHERE, "box": gc.PRIM_BOX}
OP = {"none": gc.OP_NONE, "intersect": gc.OP_INTERSECT, "union": gc.OP_UNION,
      "subtract": gc.OP_SUBTRACT}
BOOL_OP = {"union": gc.BOOL_UNION, "diff": gc.BOOL_DIFF, "intersect": gc.BOOL_INTERSECT}
BOOL_MODE = {"plain": 0, "fixed": gc.BOOL_FIXED, "dynamic": gc.BOOL_DYNAMIC}
# surface area of one period cube of each minimal surface, in squared periods
AREA = {"gyroid": 3.0915, "schwarz_p": 2.3451, "diamond": 3.8378}


def _step(name, n, tpms, period0, period1=0.0, rot=False, bend=False, modes=False, sheet=True,
          prim="none", op="none", signs=True):
    c = dict(kind="step", nx=n[0], ny=n[1], nz=n[2], tpms=tpms, period0=period0,
             period1=period1 or period0, rot=rot, bend=bend, modes=modes, sheet=sheet, prim=prim,
             op=op, signs=signs)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest edit request a server of designs sees: latency and launches
        _step("edit_40", (40, 40, 40), "gyroid", 14.0, prim="box", op="intersect"),
        # one uniform lattice cell block, the plain method's grid
        _step("plain_gyroid_128", (128, 128, 128), "gyroid", 32.0),
        # a part's bounding box (no axis a multiple of 64) with a graded, rotated lattice and
        # a hole; the caller keeps no sign words, as with a field of its own
        _step("graded_part_203", (203, 149, 181), "diamond", 14.0, 37.0, rot=True, modes=True,
              prim="sphere", op="subtract", signs=False),
        # the headline grid: everything varies
        _step("varying_schwarz_p_512", (512, 512, 512), "schwarz_p", 16.0, 64.0, rot=True,
              modes=True, prim="sphere", op="intersect"),
        # the largest grid: a bent solid lattice fused with a plate
        _step("bent_diamond_1024", (1024, 1024, 1024), "diamond", 24.0, bend=True, sheet=False,
              prim="box", op="union"),
        # a catalogue of lattice blocks evaluated and meshed per replay
        dict(name="batch_256", kind="batch", count=256, lo=32, hi=256, layout=0xBA7C),
        # a burst of edits arriving together at an interactive server
        dict(name="serve_16", kind="serve", count=16, median=96, layout=0x5E7E),
        # the reference application's largest fine grid
        dict(name="dropin_lattice_240", kind="lattice", nx=240, ny=240, nz=240, period=30.0),
        # trimming a lattice with a turned cuboid on an odd grid
        dict(name="dropin_boolean_211", kind="boolean", nx=211, ny=193, nz=229, period=30.0,
             op="intersect", mode="fixed", prim="cuboid"),
        # the reference application's largest coarse grid
        dict(name="synth_120", kind="synth", nx=120, ny=120, nz=120, period=30.0, lattice="b"),
        # a few harmonics of the reference's loop, the user's box not a cube
        dict(name="harmonics_61", kind="harmonic", nx=61, ny=57, nz=70, period=21.0, lattice="r",
             harmonics=3),
        # the reference's unit cell
        dict(name="unit_cell_61", kind="unit", n=61, cell=0),
    ]


def _size(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi], odd as often as even."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _near(rng, n, lo, hi):
    return max(lo, min(hi, int(n * rng.uniform(0.75, 1.3))))


def draw(rng):
    kind = rng.choice(["step"] * 6 + ["batch", "serve", "lattice", "boolean", "synth", "harmonic",
                                      "unit"])
    if kind == "step":
        n = _size(rng, 32, 512)
        dims = (n, _near(rng, n, 24, 640), _near(rng, n, 24, 640))
        if rng.random() < 0.3:
            dims = (max(32, n // 8 * 8),) * 3
        tpms = rng.choice(sorted(TPMS))
        period0 = round(rng.uniform(10.0, 48.0), 2)
        form = rng.choice(["uniform", "uniform", "graded", "rotated", "bent"])
        prim = rng.choice(sorted(PRIM))
        op = "none" if prim == "none" else rng.choice(["intersect", "union", "subtract"])
        return _step("", dims, tpms, period0,
                     round(rng.uniform(10.0, 64.0), 2) if form in ("graded", "rotated") else 0.0,
                     rot=form == "rotated", bend=form == "bent", modes=rng.random() < 0.4,
                     sheet=rng.random() < 0.8, prim=prim, op=op, signs=rng.random() < 0.7)
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(4, 200), lo=32, hi=rng.choice([64, 128, 192, 256]),
                    layout=rng.randrange(1 << 16))
    if kind == "serve":
        return dict(kind=kind, count=rng.randint(1, 20), median=rng.choice([48, 64, 96, 128]),
                    layout=rng.randrange(1 << 16))
    if kind in ("lattice", "boolean"):
        n = _size(rng, 24, 236)
        c = dict(kind=kind, nx=n, ny=_near(rng, n, 20, 244), nz=_near(rng, n, 20, 244),
                 period=round(rng.uniform(14.0, 40.0), 1))
        if kind == "boolean":
            c.update(op=rng.choice(sorted(BOOL_OP)), mode=rng.choice(sorted(BOOL_MODE)),
                     prim=rng.choice(["sphere", "cuboid", "torus"]))
        return c
    if kind == "synth":
        n = _size(rng, 20, 110)
        return dict(kind=kind, nx=n, ny=_near(rng, n, 16, 120), nz=_near(rng, n, 16, 120),
                    period=round(rng.uniform(12.0, 40.0), 1), lattice=rng.choice("nbrs"))
    if kind == "harmonic":
        n = _size(rng, 20, 110)
        return dict(kind=kind, nx=n, ny=_near(rng, n, 16, 120), nz=_near(rng, n, 16, 120),
                    period=round(rng.uniform(12.0, 40.0), 1), lattice=rng.choice("nbrs"),
                    harmonics=rng.randint(1, 4))
    return dict(kind="unit", n=rng.randint(24, 61), cell=rng.randint(0, 5))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _lattice_params(case, seed):
    """The grid of a step: the case's form, with the parameters an edit moves (period,
    thickness, Fourier modes, the primitive's place) from the seed; seed 0 is the design
    before any edit."""
    r = random.Random(seed)
    edit = 1.0 if seed else 0.0
    jitter = 1.0 + edit * r.uniform(-0.03, 0.03)
    t0 = (0.4 if case["modes"] else 0.3) + edit * r.uniform(-0.03, 0.03)
    bent = case["bend"]
    return CF.make(case["nx"], case["ny"], case["nz"], TPMS[case["tpms"]],
                   case["period0"] * jitter, case["period1"] * jitter, rot0=0.0,
                   rot1=math.pi / 2 if case["rot"] else 0.0, bend_radius=2.0 if bent else 0.0,
                   sheet=case["sheet"], t0=t0,
                   modes=CF.fourier_modes(seed) if case["modes"] else (), prim=PRIM[case["prim"]],
                   op=OP[case["op"]], center=tuple(0.5 + edit * r.uniform(-0.02, 0.02) for _ in range(3)),
                   radius=0.45 if case["op"] == "intersect" else 0.25,
                   half=(0.45, 0.45, 0.1 if case["op"] != "intersect" else 0.4))


def _batch_grids(case, seed):
    layout, r = CF.SplitMix64(case["layout"]), CF.SplitMix64(seed)
    sizes = list(range(case["lo"], case["hi"] + 1, 8))
    out = []
    for _ in range(case["count"]):
        nx, ny, nz = (sizes[layout.randint(len(sizes))] for _ in range(3))
        tpms = sorted(TPMS.values())[layout.randint(3)]
        period = layout.uniform(8.0, 48.0) * r.uniform(0.97, 1.03)
        out.append(CF.make(nx, ny, nz, tpms, period, sheet=True, t0=r.uniform(0.1, 0.5)))
    return out


def _requests(case, seed):
    layout, r = CF.SplitMix64(case["layout"]), CF.SplitMix64(seed)
    out = []
    for _ in range(case["count"]):
        edge = math.exp(math.log(case["median"]) + 0.5 * layout.normal())
        edge = max(16, int(round(min(384.0, edge) / 8.0)) * 8)
        tpms = sorted(TPMS.values())[layout.randint(3)]
        period = layout.uniform(8.0, 48.0) * r.uniform(0.97, 1.03)
        op = (gc.OP_INTERSECT, gc.OP_UNION, gc.OP_SUBTRACT)[layout.randint(3)]
        if layout.randint(2) == 0:
            prim = dict(prim=gc.PRIM_SPHERE, radius=r.uniform(0.35, 0.45))
        else:
            prim = dict(prim=gc.PRIM_BOX, half=(r.uniform(0.3, 0.4),) * 2 + (r.uniform(0.2, 0.4),))
        c = tuple(r.uniform(0.45, 0.55) for _ in range(3))
        out.append(CF.make(edge, edge, edge, tpms, period, sheet=True, t0=r.uniform(0.1, 0.5),
                           op=op, center=c, **prim))
    return out


def _capacity(grids):
    """Vertices to make room for: the lattices' surface area and headroom."""
    names = {v: k for k, v in TPMS.items()}
    return sum(int(1.8 * _mesh(g.npoints(), names[g.tpms], g.period0, True)[0]) + 16384
               for g in grids)


def _axes(nx, ny, nz):
    z, y, x = (torch.arange(n, dtype=torch.float64, device="cuda") for n in (nz, ny, nx))
    return x.view(1, 1, -1), y.view(1, -1, 1), z.view(-1, 1, 1)


def _grating_field(case, seed):
    """A field as the synthesis leaves it: a few gratings of a bent lattice."""
    nx, ny, nz, r = case["nx"], case["ny"], case["nz"], random.Random(seed)
    x, y, z = _axes(nx, ny, nz)
    k = 2 * math.pi / (case["period"] * (1 + r.uniform(-0.03, 0.03)))
    a = math.pi / 6 * (x / nx + y / ny)
    u, v, w = k * (x * torch.cos(a) - y * torch.sin(a)), k * (x * torch.sin(a) + y * torch.cos(a)), k * z
    p = [r.uniform(0, 2 * math.pi) for _ in range(3)]
    f = (torch.cos(u + p[0]) * torch.sin(v + p[1]) + torch.cos(v + p[1]) * torch.sin(w + p[2]) +
         torch.cos(w + p[2]) * torch.sin(u + p[0]))
    return f.float().reshape(-1).contiguous()


class _DropinBuffers:
    """The buffers the reference application allocates for a grid."""

    def __init__(self, nx, ny, nz):
        n, cells = nx * ny * nz, (nx - 1) * (ny - 1) * (nz - 1)
        self.cells, self.max_verts = cells, max(4 * n, 300000)
        self.u = {k: torch.zeros(cells, dtype=torch.int32, device="cuda")
                  for k in ("verts", "verts_scan", "occ", "occ_scan", "comp")}
        self.pos = torch.zeros((self.max_verts, 4), dtype=torch.float32, device="cuda")
        self.norm = torch.zeros_like(self.pos)
        self.grid = (gc.Uint3(nx, ny, nz), gc.Uint3(1, nx - 1, (nx - 1) * (ny - 1)),
                     gc.Uint3(nx - 1, ny - 1, nz - 1))
        self.active, self.total, self.nfacets = C.c_uint32(0), C.c_uint32(0), C.c_uint64(0)

    def arrays(self):
        return tuple(gc.ptr(self.u[k]) for k in ("verts", "verts_scan", "occ", "occ_scan"))

    def outputs(self):
        return dict(self.u, pos=self.pos, norm=self.norm, active=self.active.value,
                    total=self.total.value)


def _cuboid(case, seed):
    """Centre, angles and widths (or radii) of the primitive, in voxels from the grid's centre."""
    r = random.Random(seed)
    n = min(case["nx"], case["ny"], case["nz"])
    return dict(center=tuple(r.uniform(-0.05, 0.05) * n for _ in range(3)),
                angles=tuple(r.uniform(0.0, 1.0) for _ in range(3)),
                width=tuple(r.uniform(0.5, 0.7) * n for _ in range(3)))


def _svl_params(case, seed):
    p = gc.svl_params(case["nx"], lattice_type=case["lattice"], uniform_type=0,
                      const_period=case["period"] * (1 + random.Random(seed).uniform(-0.03, 0.03)))
    p.ny, p.nz, p.fy, p.fz = case["ny"], case["nz"], 2 * case["ny"], 2 * case["nz"]
    return p


def _coeffs(seed):
    """Coefficients of a unit cell's 5^3 Fourier series (in the reference's order)."""
    r = random.Random(seed)
    c = [complex(r.uniform(-1, 1), r.uniform(-1, 1)) /
         (1 + 2 * sum(abs(v) for v in _ijk(h))) for h in range(125)]
    return torch.tensor(c, dtype=torch.complex128).to(torch.complex64).cuda()


def _ijk(h):
    return h % 5 - 2, (h // 5) % 5 - 2, h // 25 - 2


# ---------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------
def prepare(case, seed):
    gc.init(0)
    kind = case["kind"]
    s = dict(case=case, kind=kind)
    if kind == "step":
        p = _lattice_params(case, seed)
        s["p"] = p
        s["field"] = torch.zeros(p.npoints(), dtype=torch.float32, device="cuda")
        # mesh buffers with headroom over the design before the edit
        base = _lattice_params(case, 0)
        m = gc.extract(gc.lattice_field(base, out=s["field"]), p.nx, p.ny, p.nz)
        vcap, tcap = (int(1.3 * n) + 8192 for n in (m.n_vertices, m.n_triangles))
        del m
        words = gc.sign_words(p.nx, p.ny, p.nz)
        s["signs"] = torch.zeros(words, dtype=torch.int64, device="cuda") if case["signs"] else None
        s["ws"] = torch.zeros(gc.extract_workspace_bytes(p.nx, p.ny, p.nz), dtype=torch.uint8,
                              device="cuda")
        s["vertices"] = torch.zeros((vcap, 3), dtype=torch.float32, device="cuda")
        s["triangles"] = torch.zeros((tcap, 3), dtype=torch.int32, device="cuda")
        s["counts"] = torch.zeros(2, dtype=torch.int64, device="cuda")
        a = gc.ExtractArgs()
        a.field, a.signs = s["field"].data_ptr(), s["signs"].data_ptr() if case["signs"] else None
        a.nx, a.ny, a.nz, a.iso = p.nx, p.ny, p.nz, 0.0
        a.origin = gc.Float3(0, 0, 0)
        a.spacing = gc.Float3(1 / (p.nx - 1), 1 / (p.ny - 1), 1 / (p.nz - 1))
        a.vertices, a.vert_capacity = s["vertices"].data_ptr(), vcap
        a.triangles, a.tri_capacity = s["triangles"].data_ptr(), tcap
        a.workspace, a.workspace_bytes = s["ws"].data_ptr(), s["ws"].numel()
        a.d_counts = s["counts"].data_ptr()
        s["args"] = a
    elif kind == "batch":
        vcap = _capacity(_batch_grids(case, 0))
        b = gc.Batch(_batch_grids(case, seed), use_graph=True, vert_capacity=vcap,
                     tri_capacity=2 * vcap)
        b.vertices.zero_()
        b.triangles.zero_()
        b.run()
        b.results()  # (raises when a mesh does not fit)
        s["batch"] = b
    elif kind == "serve":
        s["requests"] = _requests(case, seed)
        s["server"] = gc.Server(8 << 30)
        vcap = _capacity(_requests(case, 0))
        s["vertices"] = torch.zeros((vcap, 3), dtype=torch.float32, device="cuda")
        s["triangles"] = torch.zeros((2 * vcap, 3), dtype=torch.int32, device="cuda")
    elif kind == "lattice":
        n = case["nx"] * case["ny"] * case["nz"]
        s["svl"] = _grating_field(case, seed)
        s["ind"], s["nrm"], s["zeros"] = (torch.zeros(n, dtype=torch.float32, device="cuda")
                                          for _ in range(3))
        s["buf"] = _DropinBuffers(case["nx"], case["ny"], case["nz"])
    elif kind == "boolean":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        s["prim"] = _cuboid(case, seed)
        f = _grating_field(case, seed)
        s["lat"] = (f - f.min()) / (f.max() - f.min())
        x, y, z = _axes(nx, ny, nz)
        part = (x - 0.5 * nx) ** 2 + (y - 0.45 * ny) ** 2 + (z - 0.5 * nz) ** 2 < (0.4 * nx) ** 2
        g = torch.zeros((nx * ny * nz, 4), dtype=torch.int32, device="cuda")
        g[:, 0] = torch.where(part.reshape(-1), -1, 1).int()
        s["points0"], s["points"] = g, torch.zeros_like(g)
        s["dyn"] = torch.zeros(nx * ny * nz, dtype=torch.float32, device="cuda")
        s["buf"] = _DropinBuffers(nx, ny, nz)
    elif kind == "synth":
        s["p"], s["coeffs"] = _svl_params(case, seed), _coeffs(seed)
    elif kind == "harmonic":
        p = _svl_params(case, seed)
        n, fn = p.nx * p.ny * p.nz, p.fx * p.fy * p.fz
        s["p"], s["coeffs"] = p, _coeffs(seed)
        s["phi"] = torch.zeros(n, dtype=torch.float32, device="cuda")
        s["grating"] = torch.zeros(2 * fn, dtype=torch.float32, device="cuda")
        s["svl"] = torch.zeros(fn, dtype=torch.float32, device="cuda")
    else:
        n = case["n"]
        s["type"] = (case["cell"] + seed) % 6
        s["cell"], s["ind"], s["nrm"], s["sum"] = (
            torch.zeros(n ** 3, dtype=torch.float32, device="cuda") for _ in range(4))
        s["half"] = torch.zeros((n, n, 2 * (n // 2 + 1)), dtype=torch.float32, device="cuda")
        s["full"] = torch.zeros(2 * n ** 3, dtype=torch.float32, device="cuda")
        s["buf"] = _DropinBuffers(n, n, n)
        gc.check(gc.lib.gpucad_fft_plan3d(n, n, n))
    return s


# ---------------------------------------------------------------------------
# run
# ---------------------------------------------------------------------------
def _run_step(s):
    gc.lattice_field(s["p"], out=s["field"], signs=s["signs"])
    gc.check(gc.lib.gpucad_extract(C.byref(s["args"]), None, gc.stream_handle()))
    return dict(field=s["field"], vertices=s["vertices"], triangles=s["triangles"],
                counts=s["counts"])


def _held(t, owner):
    """`t`, a view of memory that `owner` frees, as a tensor that keeps its owner."""
    t = t.view_as(t)
    t.owner = owner
    return t


def _run_batch(s):
    b = s["batch"]
    b.run()
    return dict(fields=_held(b.fields, b), vertices=_held(b.vertices, b),
                triangles=_held(b.triangles, b))


def _run_serve(s):
    srv, reqs = s["server"], s["requests"]
    tickets = {srv.submit(p): i for i, p in enumerate(reqs)}
    done = {}
    while len(done) < len(reqs):
        for r in srv.poll():
            if r.status != gc.OK:
                raise gc.GpucadError(r.status, "request refused")
            done[tickets[r.ticket]] = r
    # the client gathers the meshes; the fields stay where they are (the arena is not carved
    # again before the next burst)
    fields, verts, tris = zip(*(srv.result_tensors(done[i], p) for i, p in enumerate(reqs)))
    torch.cat(verts, out=s["vertices"][:sum(v.shape[0] for v in verts)])
    torch.cat(tris, out=s["triangles"][:sum(t.shape[0] for t in tris)])
    torch.cuda.current_stream().synchronize()
    for r in done.values():
        srv.release(r.ticket)
    return dict(fields=[_held(f, srv) for f in fields], vertices=s["vertices"],
                triangles=s["triangles"])


def _run_lattice(s):
    c, b = s["case"], s["buf"]
    gc.check(gc.lib.gpucad_normalise_four(gc.ptr(s["svl"]), gc.ptr(s["ind"]), gc.ptr(s["nrm"]),
                                          s["svl"].numel(), c["nx"], c["ny"], c["nz"], 0.2, 0.3))
    gc.check(gc.lib.gpucad_compute_isosurface_lattice(
        gc.ptr(s["ind"]), gc.ptr(b.pos), gc.ptr(b.norm), 0.25, b.cells, *b.arrays(), *b.grid,
        gc.Float3(0.5, 0.5, 0.5), gc.Float3(0, 0, 0), C.byref(b.active), C.byref(b.total),
        gc.ptr(b.u["comp"]), b.max_verts, gc.ptr(s["nrm"]), gc.ptr(s["zeros"]), 0.2, 0.3, 0.0, 0.0))
    return dict(b.outputs(), ind=s["ind"], nrm=s["nrm"])


def _run_boolean(s):
    c, b, q = s["case"], s["buf"], s["prim"]
    flags = BOOL_OP[c["op"]] | BOOL_MODE[c["mode"]]
    n = (c["nx"], c["ny"], c["nz"], 1.0, 1.0, 1.0)
    ce, an, w = gc.Float3(*q["center"]), gc.Float3(*q["angles"]), q["width"]
    if c["mode"] != "dynamic":
        if c["prim"] == "sphere":
            st = gc.lib.gpucad_sphere_with_center(gc.ptr(s["dyn"]), ce, 0.6 * w[0], 0.0, *n, 0)
        elif c["prim"] == "cuboid":
            st = gc.lib.gpucad_cuboid(gc.ptr(s["dyn"]), ce, an, *w, *n)
        else:
            st = gc.lib.gpucad_torus_with_center(gc.ptr(s["dyn"]), ce, an, 0.5 * w[0], 0.2 * w[1],
                                                 *n)
        gc.check(st)
    s["points"].copy_(s["points0"])  # the part as it was before this edit
    gc.check(gc.lib.gpucad_classify_copy_voxel(gc.ptr(s["points"]), gc.ptr(s["dyn"]),
                                               gc.ptr(s["lat"]), b.grid[0], 0.35, 0.65, 0.0, flags))
    gc.check(gc.lib.gpucad_compute_isosurface(
        gc.ptr(b.pos), gc.ptr(b.norm), 0.0, b.cells, *b.arrays(), *b.grid,
        gc.Float3(0.5, 0.5, 0.5), gc.Float3(0, 0, 0), C.byref(b.active), C.byref(b.total),
        gc.ptr(b.u["comp"]), b.max_verts, gc.ptr(s["points"]), gc.ptr(s["dyn"]), gc.ptr(s["lat"]),
        0.35, 0.65, flags, C.byref(b.nfacets)))
    return dict(b.outputs(), dyn=s["dyn"], points=s["points"])


def _run_synth(s):
    svl, res = gc.svl_field(s["p"], s["coeffs"])
    return dict(svl=svl, iters=list(res.cg_iters), res=list(res.cg_res))


def _run_harmonic(s):
    p, lib = s["p"], gc.lib
    dims, fine = (p.nx, p.ny, p.nz), (p.fx, p.fy, p.fz)
    fn = s["svl"].numel()
    it, res = C.c_int32(0), C.c_float(0)
    iters = []
    s["svl"].zero_()
    for h in range(s["case"]["harmonics"]):
        gc.check(lib.gpucad_svl_finding_phi(gc.ptr(s["phi"]), None, *dims, *_ijk(h), 1.0, 1.0, 1.0,
                                            p.lattice_type, 0, p.const_period, 30.0, 30.0, 30.0,
                                            p.lcon, p.lcon_1, 0))
        gc.check(lib.gpucad_svl_cg(gc.ptr(s["phi"]), *dims, 500, 0.01, C.byref(it), C.byref(res)))
        iters.append(it.value)
        gc.check(lib.gpucad_svl_grating(gc.ptr(s["phi"]), *dims, gc.ptr(s["grating"]), *fine, 0.5,
                                        0.5, 0.5))
        gc.check(lib.gpucad_svl_accumulate(gc.ptr(s["svl"]), gc.ptr(s["grating"]), fn, h,
                                           gc.ptr(s["coeffs"])))
    return dict(phi=s["phi"], grating=s["grating"], svl=s["svl"], iters=iters)


def _run_unit(s):
    n, b, lib = s["case"]["n"], s["buf"], gc.lib
    gc.check(lib.gpucad_create_lattice(gc.ptr(s["cell"]), n, n, n, n ** 3, s["type"]))
    s["half"][:, :, :n].copy_(s["cell"].view(n, n, n))
    gc.check(lib.gpucad_fft_r2c(gc.ptr(s["half"])))
    gc.check(lib.gpucad_fft_scale(gc.ptr(s["half"]), float(n ** 3), n * n * (n // 2 + 1)))
    gc.check(lib.gpucad_fft_fill(gc.ptr(s["half"]), gc.ptr(s["full"]), n, n, n))
    gc.check(lib.gpucad_fft_c2c_inverse(gc.ptr(s["full"])))
    s["sum"].zero_()
    gc.check(lib.gpucad_grating_sum(gc.ptr(s["full"]), gc.ptr(s["sum"]), n, n, n))
    coeffs = gc.unit_spectrum(s["cell"], n, 2)
    gc.check(lib.gpucad_normalise_four(gc.ptr(s["cell"]), gc.ptr(s["ind"]), gc.ptr(s["nrm"]),
                                       n ** 3, n, n, n, 0.2, 0.3))
    gc.check(lib.gpucad_compute_isosurface_latticeone(
        gc.ptr(s["ind"]), gc.ptr(b.pos), gc.ptr(b.norm), 0.25, b.cells, *b.arrays(), *b.grid,
        gc.Float3(1, 1, 1), gc.Float3(0, 0, 0), C.byref(b.active), C.byref(b.total),
        gc.ptr(b.u["comp"]), b.max_verts, gc.ptr(s["nrm"]), 0.2, 0.3))
    return dict(b.outputs(), cell=s["cell"], half=s["half"], wave=s["full"], sum=s["sum"],
                coeffs=coeffs, ind=s["ind"], nrm=s["nrm"])


def run(state):
    return globals()["_run_" + state["kind"]](state)


# ---------------------------------------------------------------------------
# work: each input read once, each output written once (mesh sizes estimated
# from the surface's area: 3/2 crossing edges per unit area, two triangles per
# vertex)
# ---------------------------------------------------------------------------
def _mesh(points, tpms, period, sheet, share=1.0):
    v = 1.5 * AREA[tpms] * (2 if sheet else 1) * points / period * share
    return v, 2 * v


def work(case):
    kind = case["kind"]
    if kind == "step":
        n = case["nx"] * case["ny"] * case["nz"]
        p0, p1 = case["period0"], case["period1"]
        period = p0 if p0 == p1 else (p1 - p0) / math.log(p1 / p0)
        share = 0.4 if case["op"] == "intersect" else 0.9
        v, t = _mesh(n, case["tpms"], period, case["sheet"], share)
        per_point = (140 if case["rot"] or case["bend"] else 82) + (155 if case["modes"] else 0)
        return dict(bytes=4 * n + 12 * (v + t), flops=per_point * n)
    if kind == "batch":
        grids = _batch_grids(case, 0)
        n = sum(g.npoints() for g in grids)
        v = sum(_mesh(g.npoints(), "gyroid", g.period0, True)[0] for g in grids)
        return dict(bytes=4 * n + 36 * v, flops=82 * n)
    if kind == "serve":
        grids = _requests(case, 0)
        n = sum(g.npoints() for g in grids)
        v = sum(_mesh(g.npoints(), "gyroid", g.period0, True, 0.6)[0] for g in grids)
        return dict(bytes=4 * n + 36 * v, flops=92 * n)
    if kind in ("lattice", "boolean"):
        n = case["nx"] * case["ny"] * case["nz"]
        v, t = _mesh(n, "gyroid", case["period"], True, 0.9 if kind == "lattice" else 0.3)
        # lattice: field in, indicator and normalised out, five uint arrays; boolean: the
        # primitive out, grid_points in and out, the lattice in, five uint arrays; float4
        # position and normal per corner
        return dict(bytes=((4 + 8) if kind == "lattice" else (4 + 32 + 4)) * n + 16 * n + 96 * t,
                    flops=40 * n)
    if kind in ("synth", "harmonic"):
        n = case["nx"] * case["ny"] * case["nz"]
        if kind == "synth":  # the fine field out; three solves of about 2 max(n) iterations
            it = 2 * max(case["nx"], case["ny"], case["nz"])
            return dict(bytes=4 * 8 * n, flops=3 * it * 30 * n + 62 * 20 * 8 * n)
        it = 2 * max(case["nx"], case["ny"], case["nz"]) * case["harmonics"]
        return dict(bytes=(4 * n + 20 * 8 * n) * case["harmonics"], flops=it * 30 * n)
    n = case["n"] ** 3
    v, t = _mesh(n, "gyroid", case["n"], True)
    return dict(bytes=(4 * 4 + 8 * 2 + 20) * n + 96 * t, flops=2 * 15 * n * math.log2(n))


# ---------------------------------------------------------------------------
# exact: the computed numbers in 64 bits, in plain torch (mesh vertices and
# normals have no such value: which edges they lie on follows from the field's
# own bits)
# ---------------------------------------------------------------------------
def _exact_field(p):
    nx, ny, nz = p.nx, p.ny, p.nz
    out = torch.empty((nz, ny, nx), dtype=torch.float64, device="cuda")
    x, y, _ = _axes(nx, ny, nz)
    hx, hy, hz = 1.0 / (nx - 1), 1.0 / (ny - 1), 1.0 / (nz - 1)
    two_pi = 2 * math.pi
    period = p.period0 + (p.period1 - p.period0) * x * hx
    planes = max(1, (1 << 24) // (nx * ny))
    for z0 in range(0, nz, planes):
        z = torch.arange(z0, min(nz, z0 + planes), dtype=torch.float64, device="cuda").view(-1, 1, 1)
        u, v, w = x, y, z
        if p.rot0 or p.rot1:
            th = p.rot0 + (p.rot1 - p.rot0) * z * hz
            dx, dy = x - 0.5 * (nx - 1), y - 0.5 * (ny - 1)
            u = 0.5 * (nx - 1) + torch.cos(th) * dx - torch.sin(th) * dy
            v = 0.5 * (ny - 1) + torch.sin(th) * dx + torch.cos(th) * dy
        elif p.bend_radius > 0:
            ax, ay = x * hx - 0.5, y * hy - (0.5 - p.bend_radius)
            u = (0.5 + p.bend_radius * torch.atan2(ax, ay)) / hx
            v = (0.5 - p.bend_radius + torch.sqrt(ax * ax + ay * ay)) / hy
        u, v, w = two_pi * u / period, two_pi * v / period, two_pi * w / period
        sx, cx, sy, cy, sz, cz = (f(t) for t in (u, v, w) for f in (torch.sin, torch.cos))
        if p.tpms == gc.TPMS_GYROID:
            f = sx * cy + sy * cz + sz * cx
        elif p.tpms == gc.TPMS_SCHWARZ_P:
            f = cx + cy + cz
        else:
            f = sz * (sx * sy + cx * cy) + cz * (sx * cy + cx * sy)
        if p.sheet:
            t = torch.full((1, 1, 1), p.t0, dtype=torch.float64, device="cuda")
            for m in range(p.n_modes):
                k = p.mode_k[m]
                t = t + p.mode_a[m] * torch.cos(
                    two_pi * (k[0] * x * hx + k[1] * y * hy + k[2] * z * hz + p.mode_phi[m]))
            f = f.abs() - t
        q = [c * h - o for c, h, o in zip((x, y, z), (hx, hy, hz), p.prim_center)]
        if p.prim == gc.PRIM_SPHERE:
            d = torch.sqrt(q[0] ** 2 + q[1] ** 2 + q[2] ** 2) - p.prim_radius
        elif p.prim == gc.PRIM_BOX:
            b = [c.abs() - h for c, h in zip(q, p.prim_half)]
            d = (torch.sqrt(sum(c.clamp(min=0) ** 2 for c in b)) +
                 torch.maximum(torch.maximum(b[0], b[1]), b[2]).clamp(max=0))
        if p.prim != gc.PRIM_NONE:
            f = {gc.OP_INTERSECT: lambda: torch.maximum(f, d), gc.OP_UNION: lambda: torch.minimum(f, d),
                 gc.OP_SUBTRACT: lambda: torch.maximum(f, -d), gc.OP_NONE: lambda: f}[p.op]()
        out[z0:z0 + z.shape[0]] = f
    return out.reshape(-1)


def _exact_primitive(case, q):
    """The primitive's implicit (Modelling's squared forms), in voxels from the grid's centre."""
    x, y, z = _axes(case["nx"], case["ny"], case["nz"])
    v = [c - 0.5 * (n - 1) - o for c, n, o in zip((x, y, z), (case["nx"], case["ny"], case["nz"]),
                                                  (C.c_float(o).value for o in q["center"]))]
    w = [C.c_float(a).value for a in q["width"]]
    if case["prim"] == "sphere":
        return (v[0] ** 2 + v[1] ** 2 + v[2] ** 2 - (0.6 * w[0]) ** 2).reshape(-1)
    (cx, sx), (cy, sy), (cz, sz) = ((math.cos(a), math.sin(a)) for a in q["angles"])
    rows = ((cz * cy, cz * sy * sx - sz * cx, cz * sy * cx + sz * sx),
            (sz * cy, sz * sy * sx + cz * cx, sz * sy * cx - cz * sx), (-sy, cy * sx, cy * cx))
    r = [v[0] * a + v[1] * b + v[2] * c for a, b, c in rows]
    if case["prim"] == "cuboid":
        d = [c.abs() - 0.5 * a for c, a in zip(r, w)]
        return torch.maximum(torch.maximum(d[0], d[1]), d[2]).reshape(-1)
    side = 0.5 * w[0] - torch.sqrt(r[0] ** 2 + r[1] ** 2)
    return (r[2] ** 2 - (0.2 * w[1]) ** 2 + side ** 2).reshape(-1)


def _gradient(n):
    """The 1-D difference the phase solve uses: central inside, one-sided at the ends."""
    g = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    i = torch.arange(1, n - 1, device="cuda")
    g[i, i - 1], g[i, i + 1] = -0.5, 0.5
    g[0, 0], g[0, 1], g[n - 1, n - 2], g[n - 1, n - 1] = -1.0, 1.0, -1.0, 1.0
    return g


def _exact_phases(p):
    """The zero-mean phases of the unit wave numbers that best fit the lattice's grating
    vectors in the least-squares sense, by the operator's 1-D eigenvectors."""
    dims = (p.nx, p.ny, p.nz)
    x, y, z = (c + 1 for c in _axes(*dims))
    k = 2 * math.pi / p.const_period
    if p.lattice_type in (b"b", b"r"):
        mx, my = ((p.nx + 1) / 2, (p.ny + 1) / 2) if p.lattice_type == b"r" else (0.0, 0.0)
        th = torch.atan2(y - my, x - mx)
    elif p.lattice_type == b"s":
        th = p.lcon * torch.sin(6.28 * p.lcon_1 * x)
    else:
        th = torch.zeros_like(x)
    one, none = torch.ones_like(x + y + z), torch.zeros_like(x + y + z)
    c, s = torch.cos(th) * one, torch.sin(th) * one
    grads = [_gradient(n) for n in dims]  # x, y, z
    vals, vecs = zip(*(torch.linalg.eigh(g.T @ g) for g in grads))

    def along(f, m, axis):  # m applied along an axis of f[z, y, x]
        return torch.movedim(torch.tensordot(m, f, dims=([1], [axis])), 0, axis)

    lam = vals[0].view(1, 1, -1) + vals[1].view(1, -1, 1) + vals[2].view(-1, 1, 1)
    lam[0, 0, 0] = math.inf  # the constant
    out = []
    for kx, ky, kz in ((c, s, none), (-s, c, none), (none, none, one)):
        b = sum(along(k * f, g.T, 2 - a) for a, (f, g) in enumerate(zip((kx, ky, kz), grads)))
        for a in range(3):
            b = along(b, vecs[a].T, 2 - a)
        b = b / lam
        for a in range(3):
            b = along(b, vecs[a], 2 - a)
        out.append(b)
    return out


def _refine(f):
    """Twice as fine along each axis: even points copy, odd ones average, the last repeats."""
    for a in range(3):
        nxt = torch.cat([f.narrow(a, 1, f.shape[a] - 1), f.narrow(a, f.shape[a] - 1, 1)], a)
        f = torch.stack([f, 0.5 * (f + nxt)], a + 1).flatten(a, a + 1)
    return f


def _exact_unit(case, kind):
    n = case["n"]
    x, y, z = (2.0 * c / (n - 1) - 1.0 for c in _axes(n, n, n))
    (ax, ay, az), (bx, by, bz) = ([k * c for c in (x, y, z)] for k in (3.14, 6.28))
    sin, cos = torch.sin, torch.cos
    if kind == 0:
        f = cos(ax) * sin(ay) + cos(ay) * sin(az) + cos(az) * sin(ax)
    elif kind == 1:
        f = cos(ax) + cos(ay) + cos(az)
    elif kind == 2:
        f = 4 * cos(x) * cos(y) * cos(z) - (cos(2 * x) * cos(2 * y) + cos(2 * y) * cos(2 * z) +
                                            cos(2 * z) * cos(2 * x))
    elif kind == 3:
        f = 2 * (cos(ax) * cos(ay) + cos(ay) * cos(az) + cos(az) * cos(ax)) - (cos(bx) + cos(by) +
                                                                               cos(bz))
    elif kind == 4:
        f = torch.minimum(torch.minimum(x * x + y * y, y * y + z * z), z * z + x * x)
    else:
        f = cos(ax) * cos(ay) * cos(az) - sin(ax) * sin(ay) * sin(az)
    return f


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return dict(field=_exact_field(_lattice_params(case, seed)), vertices=None, triangles=None,
                    counts=None)
    if kind == "batch":
        return dict(fields=torch.cat([_exact_field(g) for g in _batch_grids(case, seed)]),
                    vertices=None, triangles=None)
    if kind == "serve":
        return dict(fields=[_exact_field(g) for g in _requests(case, seed)], vertices=None,
                    triangles=None)
    mesh = dict.fromkeys(("verts", "verts_scan", "occ", "occ_scan", "comp", "pos", "norm", "active",
                          "total"))
    if kind in ("lattice", "unit"):
        shape = (case["n"],) * 3 if kind == "unit" else (case["nz"], case["ny"], case["nx"])
        f = _exact_unit(case, (case["cell"] + seed) % 6) if kind == "unit" else \
            _grating_field(case, seed).double().view(shape)
        lo, hi = f.min().clamp(max=0), f.max().clamp(min=0)
        nrm = torch.zeros_like(f)
        nrm[1:-1, 1:-1, 1:-1] = ((f - lo) / (hi - lo))[1:-1, 1:-1, 1:-1]
        out = dict(mesh, ind=None, nrm=nrm.reshape(-1))
        if kind == "lattice":
            return out
        n = case["n"]
        half = torch.fft.rfftn(f) / n ** 3
        pick = [v % n for v in range(-2, 3)]
        full = torch.fft.fftn(f) / n ** 3
        wave = torch.view_as_real(f + 0j).reshape(-1)
        return dict(out, cell=f.reshape(-1), half=torch.view_as_real(half).reshape(n, n, -1),
                    wave=wave, sum=f.reshape(-1),
                    coeffs=full[pick][:, pick][:, :, pick].reshape(-1))
    if kind == "boolean":
        dyn = torch.zeros(case["nx"] * case["ny"] * case["nz"], dtype=torch.float64)
        if case["mode"] != "dynamic":
            dyn = _exact_primitive(case, _cuboid(case, seed))
        return dict(mesh, dyn=dyn, points=None)
    # the synthesis stops at a residual, so its outputs lie near these
    p, coeffs = _svl_params(case, seed), _coeffs(seed).to(torch.complex128)
    phases = _exact_phases(p)
    fine = [_refine(f) for f in phases]
    count = case["harmonics"] if kind == "harmonic" else p.harmonics
    svl = torch.zeros_like(fine[0])
    for h in range(count):
        wave = torch.polar(torch.ones_like(svl), sum(m * f for m, f in zip(_ijk(h), fine)))
        svl += (wave * coeffs[h]).real
    if kind == "synth":
        return dict(svl=svl.reshape(-1), iters=None, res=None)
    phi = sum(m * f for m, f in zip(_ijk(count - 1), phases))
    return dict(phi=phi.reshape(-1), grating=torch.view_as_real(wave).reshape(-1),
                svl=svl.reshape(-1), iters=None)

"""The calls a CFD code makes of this library, at the sizes it makes them, for timing.

Every case is one pass through public entry points: the drop-in solver call on host arrays, the
resident pressure solves (FP64 and learned), the momentum solves, the calls of a SIMPLE step with
fields in device memory, and the forward and backward pass of network training.  Meshes are the
families the benchmark and the tests use: hexahedral boxes with interior vertices perturbed by 20 %
(optionally graded by 1.05 toward x = 0, cells up to 100 times thinner than wide) and permuted
Kuhn tetrahedra graded by 1.1.

`exact` evaluates the same quantities in 64 bits with plain torch: geometry, matrix, gradients and
fluxes from the mesh's points, solves by Jacobi-preconditioned CG far below the solvers' tolerance.
"""
import functools
import math

import numpy as np
import torch

from freecappuccino_amd import fcap, gnn
from freecappuccino_amd import mesh as M

SOLVE_TOL = 1e-8      # the tolerance the benchmark solves to
VIS, URF = 1e-3, 0.7  # viscosity and under-relaxation of the momentum systems
BLOBS = 16            # Gaussian blobs in a right-hand side

METHODS = {"iccg": fcap.METHOD_ICCG, "dpcg": fcap.METHOD_DPCG, "bicgstab": fcap.METHOD_BICGSTAB,
           "bicgstab_mixed": fcap.METHOD_BICGSTAB_MIXED, "fcg_learned": fcap.METHOD_FCG_LEARNED,
           "fcg_jacobi": fcap.METHOD_FCG_JACOBI}


def _box(name, kind, nx, ny, nz, graded=False, method=""):
    return {"name": name, "kind": kind, "mesh": "box", "nx": nx, "ny": ny, "nz": nz, "graded": graded,
            "method": method}


def _tets(name, kind, n, method=""):
    return {"name": name, "kind": kind, "mesh": "tets", "nx": n, "ny": n, "nz": n, "graded": True, "method": method}


def listed():
    return [
        # the reference's own solver call, host arrays in and out, on its cavity example's 20 x 20 cells
        _box("host_iccg_cavity", "host_solve", 20, 20, 1, method="iccg"),
        # one pressure correction of a SIMPLE iteration on the reference's backward-facing-step size
        # (about 12 thousand cells, two-dimensional), fields resident
        _box("simple_step_2d", "simple", 163, 75, 1, method="iccg"),
        # DIC-PCG on the 40^3 box of the parity tests
        _box("iccg_40", "solve", 40, 40, 40, method="iccg"),
        # DIC-PCG on the perturbed 128^3 box the benchmark times
        _box("iccg_128", "solve", 128, 128, 128, method="iccg"),
        # Jacobi-PCG on a box with no round edge
        _box("dpcg_97x83x61", "solve", 97, 83, 61, method="dpcg"),
        # momentum on the benchmark's permuted graded tetrahedra, FP64 BiCGStab
        _tets("momentum_tets_24", "momentum", 24, method="bicgstab"),
        # the three momentum components on a graded box in mixed precision
        _box("momentum_mixed_96x80x72", "momentum", 96, 80, 72, True, "bicgstab_mixed"),
        # the benchmark's headline solve: learned flexible CG on the graded 192^3 box
        _box("fcg_learned_192", "solve", 192, 192, 192, True, "fcg_learned"),
        # the same flexible CG without the network, the fastest solver of a static matrix
        _box("fcg_jacobi_128", "solve", 128, 128, 128, method="fcg_jacobi"),
        # gradients and pressure-correction assembly at the largest size
        _box("assemble_192", "assemble", 192, 192, 192, True),
        # corrections and the non-orthogonal corrector's source, ragged
        _box("correct_151x93x77", "correct", 151, 93, 77, True),
        # forward and backward pass of training on the 64^3 systems it streams
        _box("network_grad_64", "network_grad", 64, 64, 64),
    ]


# Cells a drawn case of each kind may have, and the methods its kind is used with.
_DRAWN = [
    ("host_solve", 100, 30_000, ("iccg", "bicgstab")),
    ("simple", 400, 500_000, ("iccg", "dpcg")),
    ("solve", 1_000, 2_000_000, ("iccg", "dpcg")),
    ("solve", 8_000, 3_500_000, ("fcg_learned", "fcg_jacobi")),
    ("momentum", 1_000, 600_000, ("bicgstab", "bicgstab_mixed")),
    ("assemble", 400, 7_000_000, ("",)),
    ("correct", 400, 7_000_000, ("",)),
    ("network_grad", 1_000, 300_000, ("",)),
]


def _unnamed(case):
    return {k: v for k, v in case.items() if k != "name"}


def draw(rng):
    kind, lo, hi, methods = rng.choice(_DRAWN)
    cells = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    method = rng.choice(methods)
    # (the pressure correction's coefficient, as the reference writes it, vanishes on faces of such tetrahedra)
    if kind == "momentum" and cells < 150_000 and rng.random() < 0.4:
        n = max(3, round((cells / 6) ** (1 / 3)))
        return _unnamed(_tets("", kind, n, method))
    if kind in ("host_solve", "simple") and cells < 30_000 and rng.random() < 0.5:
        nx = max(3, round(math.sqrt(cells * rng.uniform(0.5, 2.0))))
        ny, nz = max(3, round(cells / nx)), 1
    else:
        side = cells ** (1 / 3)
        nx = max(3, round(side * rng.uniform(0.7, 1.4)))
        ny = max(3, round(side * rng.uniform(0.7, 1.4)))
        nz = max(2, round(cells / (nx * ny)))
    graded = nz > 1 and kind != "host_solve" and rng.random() < 0.4
    if kind == "solve" and method == "dpcg":
        graded = False   # Jacobi-PCG is not used on meshes of that aspect ratio
    return _unnamed(_box("", kind, nx, ny, nz, graded, method))


# ------------------------------------------------------------------------------------ meshes

@functools.lru_cache(maxsize=6)
def _box_topology(nx, ny, nz, inlet_outlet):
    """Faces of hex_box's mesh (cells x fastest, faces in upper-triangular order), points apart."""
    px, pxy = nx + 1, (nx + 1) * (ny + 1)
    c = torch.arange(nx * ny * nz, device="cuda")
    i, j, k = c % nx, (c // nx) % ny, c // (nx * ny)
    base = i + px * j + pxy * k
    corners = torch.tensor([[1, 1 + px, 1 + px + pxy, 1 + pxy], [px, px + pxy, 1 + px + pxy, 1 + px],
                            [pxy, 1 + pxy, 1 + px + pxy, px + pxy]], device="cuda")
    inside = torch.stack([i < nx - 1, j < ny - 1, k < nz - 1], 1)
    neighbour = (c[:, None] + torch.tensor([1, nx, nx * ny], device="cuda"))[inside]
    owner = c[:, None].expand(-1, 3)[inside]
    nodes = (base[:, None, None] + corners)[inside]
    sides = [(i == 0, [0, pxy, px + pxy, px]), (i == nx - 1, corners[0].tolist()),
             (j == 0, [0, 1, 1 + pxy, pxy]), (j == ny - 1, corners[1].tolist()),
             (k == 0, [0, px, 1 + px, 1]), (k == nz - 1, corners[2].tolist())]
    types = (["inlet", "outlet"] + ["wall"] * 4) if inlet_outlet else (["wall"] + ["symmetry"] * 5)
    patches, all_own, all_nodes, at = [], [owner], [nodes], owner.shape[0]
    for kind, (mask, corner) in zip(types, sides):
        cells = c[mask]
        all_own.append(cells)
        all_nodes.append(base[mask][:, None] + torch.tensor(corner, device="cuda"))
        patches.append((kind, cells.shape[0], at))
        at += cells.shape[0]
    to_host = lambda t: t.to(torch.int32).cpu().numpy()  # noqa: E731
    return (np.arange(0, 4 * at + 1, 4, dtype=np.int32), to_host(torch.cat(all_nodes).reshape(-1)),
            to_host(torch.cat(all_own)), to_host(neighbour), patches)


def _box_points(nx, ny, nz, graded, seed):
    """Nodes of the box in [0,1]^3, interior ones moved by up to 20 % of the smaller spacing beside them."""
    axes = [M.graded_spacing(nx, 1.05, 100.0) if graded else M.uniform_spacing(nx), M.uniform_spacing(ny),
            M.uniform_spacing(nz)]
    g = torch.Generator("cuda").manual_seed(seed)
    shape = (nz + 1, ny + 1, nx + 1)
    pts = torch.empty(shape + (3,), dtype=torch.float64, device="cuda")
    inner = torch.zeros(shape, dtype=torch.float64, device="cuda")
    inner[1:-1, 1:-1, 1:-1] = 0.2
    for a, h in enumerate(axes):
        d = np.diff(h)
        near = np.concatenate([d[:1], np.minimum(d[:-1], d[1:]), d[-1:]])
        view = [1, 1, 1]
        view[2 - a] = len(h)
        move = 2.0 * torch.rand(shape, dtype=torch.float64, device="cuda", generator=g) - 1.0
        pts[..., a] = (torch.from_numpy(h).cuda().reshape(view)
                       + inner * move * torch.from_numpy(near).cuda().reshape(view))
    return pts.reshape(-1, 3).cpu().numpy()


@functools.lru_cache(maxsize=3)
def _tet_mesh(n, inlet_outlet):
    bc = dict(x0="inlet", x1="outlet", y0="wall", y1="wall", z0="wall", z1="wall") if inlet_outlet else None
    return M.tet_box(n, grade_axis=1, grade_ratio=1.1, grade_max_aspect=100.0, permute_seed=3, bc=bc)


def _mesh(case, seed):
    inlet_outlet = case["kind"] in ("simple", "assemble", "correct")
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["mesh"] == "tets":
        return _tet_mesh(nx, inlet_outlet)
    face_ptr, nodes, owner, neighbour, patches = _box_topology(nx, ny, nz, inlet_outlet)
    return M.PolyMesh(_box_points(nx, ny, nz, case["graded"], seed), face_ptr, nodes, owner, neighbour, nx * ny * nz,
                      patches)


# ------------------------------------------------------------------------------------ inputs

class _Shared:
    """Device memory of a resident system, for torch to read without a copy."""

    def __init__(self, system, name, count):
        self.system = system   # the memory is the system's: it lives as long as the tensor
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": "<f8", "version": 2,
                                         "data": (system.device_ptr(name), False)}


def _array(system, name, count):
    tensor = torch.as_tensor(_Shared(system, name, count), device="cuda")
    tensor.owner = system
    return tensor


class _Geometry:
    """Cell and face geometry and connectivity as torch tensors."""

    def __init__(self, m, system=None):
        nf, self.nif, self.n = m.n_faces, m.n_inner, m.n_cells
        self.own = torch.from_numpy(m.owner).cuda().long()
        self.nei = torch.from_numpy(m.neighbour).cuda().long()
        self.p = self.own[:self.nif]
        first, count = m.wall_range()
        self.walls = slice(first, first + count)
        if system is None:
            self._from_points(m)
            return
        stack = lambda names, count: torch.stack([_array(system, k, count) for k in names], 1)  # noqa: E731
        self.s, self.xf = stack(("arx", "ary", "arz"), nf), stack(("xf", "yf", "zf"), nf)
        self.xc, self.vol = stack(("xc", "yc", "zc"), self.n), _array(system, "vol", self.n)
        self.fac = _array(system, "facint", self.nif)

    def _from_points(self, m):
        x = torch.from_numpy(m.points).cuda()
        node = torch.from_numpy(m.face_nodes).cuda().long().reshape(m.n_faces, -1)
        a = x[node[:, 0]]
        self.s = torch.zeros_like(a)
        self.vol = torch.zeros(self.n, dtype=torch.float64, device="cuda")
        centre = torch.zeros(self.n, 3, dtype=torch.float64, device="cuda")
        for i in range(1, node.shape[1] - 1):
            b, c = x[node[:, i]], x[node[:, i + 1]]
            area2 = torch.linalg.cross(b - a, c - a)
            self.s += 0.5 * area2
            self.sum_faces(self.vol, ((a + b + c) / 3.0 * area2).sum(1) / 6.0)
            self.sum_faces(centre, area2 / 48.0 * ((a + b) ** 2 + (b + c) ** 2 + (c + a) ** 2))
        self.xf = x[node].mean(1)
        self.xc = centre / self.vol[:, None]
        b, c = x[node[:self.nif, 1]], x[node[:self.nif, 2]]
        normal = torch.linalg.cross(b - a[:self.nif], c - a[:self.nif])
        d = self.xc[self.nei] - self.xc[self.p]
        self.fac = ((normal * (a[:self.nif] - self.xc[self.p])).sum(1) / (normal * d).sum(1)).abs()

    def sum_faces(self, out, value):
        """out(owner) += value, out(neighbour) -= value over the faces."""
        out.index_add_(0, self.own[:value.shape[0]], value)
        out.index_add_(0, self.nei, -value[:self.nif])
        return out

    def at_faces(self, value):
        w = self.fac if value.dim() == 1 else self.fac[:, None]
        return (1.0 - w) * value[self.p] + w * value[self.nei]


def _generator(seed):
    return torch.Generator("cuda").manual_seed(1_000_003 + seed)


def _rand(g, *shape):
    return torch.rand(*shape, dtype=torch.float64, device="cuda", generator=g)


def _blobs(g, geo, count=BLOBS):
    """A sum of Gaussian blobs with zero mean, times the cell volumes."""
    centre, width = _rand(g, count, 3).tolist(), (0.02 + 0.18 * _rand(g, count)).tolist()
    sign = torch.sign(_rand(g, count) - 0.5).tolist()
    f = torch.zeros(geo.n, dtype=torch.float64, device="cuda")
    for c, w, s in zip(centre, width, sign):
        r2 = sum((geo.xc[:, a] - c[a]) ** 2 for a in range(3))
        f += s * torch.exp(-r2 / (2.0 * w * w))
    f -= (f * geo.vol).sum() / geo.vol.sum()
    return f * geo.vol


def _velocity(g, geo):
    """A Taylor-Green velocity with a seeded phase."""
    x = 2.0 * math.pi * (geo.xc + _rand(g, 3))
    return torch.stack([torch.sin(x[:, 0]) * torch.cos(x[:, 1]) * torch.cos(x[:, 2]),
                        -torch.cos(x[:, 0]) * torch.sin(x[:, 1]) * torch.cos(x[:, 2]),
                        torch.zeros(geo.n, dtype=torch.float64, device="cuda")], 1)


def _step_fields(geo, seed):
    """Fields of a SIMPLE step: u, v, w, p with boundary values, density, 1/a_P, pp with boundary values."""
    g = _generator(seed)
    vel = _velocity(g, geo)
    x, phase = geo.xc, _rand(g, 2)
    p = torch.sin(3.0 * x[:, 0] + phase[0]) * x[:, 1] + x[:, 2]
    pp = 1e-2 * torch.cos(2.0 * x[:, 1] + phase[1]) * x[:, 0]
    ap = (0.5 + _rand(g, 3, geo.n)) / geo.vol
    cells = torch.stack([vel[:, 0], vel[:, 1], vel[:, 2], p, pp])
    cells = torch.cat([cells, cells[:, geo.own[geo.nif:]]], 1)
    return {"uvwp": cells[:4].contiguous(), "pp": cells[4].contiguous(), "ap": ap.contiguous(),
            "den": 1.0 + 0.1 * _rand(g, geo.n)}


def _momentum_inputs(geo, seed):
    """Mass fluxes of a Taylor-Green field, and each component's sp, source and start."""
    g = _generator(seed)
    flux = (geo.at_faces(_velocity(g, geo)) * geo.s[:geo.nif]).sum(1)
    sp = [10.0 * _rand(g, geo.n) * geo.vol for _ in range(3)]
    src = [_blobs(g, geo, 8) for _ in range(3)]
    phi = [0.2 * _rand(g, geo.n) - 0.1 for _ in range(3)]
    return flux, sp, src, phi


def _network_pair(geo, seed, op):
    """Residual and error as training meets them: noise whose rough part a smoother has damped."""
    e = 2.0 * _rand(_generator(seed), geo.n) - 1.0
    for _ in range(4):
        e = e - 0.8 * op(e) / op.diag
    return op(e).float(), e.float()


# ------------------------------------------------------------------------------------ states

_shared = {}


def _context():
    """One context for the process, on a stream that torch knows."""
    if not _shared:
        _shared["stream"] = torch.cuda.Stream()
        _shared["ctx"] = fcap.Context(0)
        _shared["ctx"].set_stream(_shared["stream"].cuda_stream)
    return _shared["ctx"]


def _address(t, row=0):
    return t.data_ptr() + 8 * row * (t.shape[-1] if t.dim() > 1 else 0)


def prepare(case, seed):
    ctx = _context()
    m = _mesh(case, seed)
    system = fcap.System(m, ctx)
    geo = _Geometry(m, system)
    kind, st = case["kind"], {"case": case, "system": system}
    host = lambda t: t.cpu().numpy()  # noqa: E731
    if kind in ("solve", "host_solve", "network_grad"):
        su = host(_blobs(_generator(seed), geo))
        system.assemble_laplacian(np.full(m.n_cells, -1.0), None, su)
        st["zero"] = np.zeros(m.n_cells)
        if case["method"] == "fcg_learned" or kind == "network_grad":
            st["net"] = gnn.Network.load(ctx=ctx)
            st["net"].attach(system)
        if kind == "host_solve":
            st["csr"] = fcap.CSR(*(system.get(k) for k in ("ioffset", "ja", "diag", "ij_slot", "ji_slot")))
            st["a"], st["su"] = system.get("a"), system.get("su")
        if kind == "network_grad":
            st["r"], st["e"] = (host(t) for t in _network_pair(geo, seed, _Operator(geo)))
    elif kind == "momentum":
        flux, sp, src, phi = _momentum_inputs(geo, seed)
        st.update(flux=host(flux), vis=np.full(m.n_cells, VIS), sp=[host(t) for t in sp],
                  src=[host(t) for t in src], phi=[host(t) for t in phi])
    else:
        st.update(_step_fields(geo, seed))
        new = lambda *shape: torch.zeros(*shape, dtype=torch.float64, device="cuda")  # noqa: E731
        st["grads"], st["flmass"] = new(4, 3 * geo.n), new(geo.nif)
        st["a"], st["rhs"] = _array(system, "a", m.nnz), _array(system, "su", geo.n)
        if kind == "simple":
            st["work"], st["dpp"] = st["uvwp"].clone(), new(3 * geo.n)
        if kind == "correct":
            _assemble(st, st["uvwp"])
            st["dpp"] = new(3 * geo.n)
    torch.cuda.synchronize()
    return st


def _assemble(st, uvwp):
    s, grads, ap = st["system"], st["grads"], st["ap"]
    for k in range(4):
        s.grad_gauss(_address(uvwp, k), 1, out=_address(grads, k))
    s.calcp_assemble(_address(st["den"]), *(_address(ap, k) for k in range(3)), *(_address(uvwp, k) for k in range(4)),
                     *(_address(grads, k) for k in range(4)), flmass=_address(st["flmass"]))


def _correct(st, uvwp, pp):
    st["system"].calcp_correct(_address(st["dpp"]), *(_address(st["ap"], k) for k in range(3)), 0.3, 0,
                               _address(st["flmass"]), *(_address(uvwp, k) for k in range(4)), pp=pp)


def run(st):
    case, s = st["case"], st["system"]
    kind = case["kind"]
    if kind == "solve":
        s.assemble_laplacian_dev()
        s.set_solution(st["zero"])
        s.solve(METHODS[case["method"]], fcap.STOP_L2, SOLVE_TOL, 20_000)
        return s.solution()
    if kind == "host_solve":
        solver = fcap.iccg if case["method"] == "iccg" else fcap.bicgstab
        return solver(st["csr"], st["a"], st["su"], st["zero"], sor=SOLVE_TOL, nsw=2_000, ctx=s.ctx).fi
    if kind == "momentum":
        s.assemble_convdiff(st["vis"], st["flux"], URF, None)
        _, phi, ap, _ = s.solve_momentum(st["sp"], st["src"], [URF] * 3, st["phi"], METHODS[case["method"]], SOLVE_TOL,
                                         2_000)
        return {"phi": phi, "ap": ap}
    if kind == "network_grad":
        loss, grad = st["net"].loss_grad(s, st["r"], st["e"])
        return {"loss": loss, "grad": grad}
    if kind == "assemble":
        _assemble(st, st["uvwp"])
        return {k: st[k] for k in ("grads", "a", "rhs", "flmass")}
    if kind == "correct":
        s.grad_gauss(_address(st["pp"]), 1, out=_address(st["dpp"]))
        _correct(st, st["uvwp"], _address(st["pp"]))
        s.calcp_nonorth(_address(st["den"]), _address(st["ap"]), _address(st["dpp"]), _address(st["flmass"]))
        return {k: st[k] for k in ("dpp", "uvwp", "flmass", "rhs")}
    # a pressure correction from the momentum predictor's fields
    with torch.cuda.stream(_shared["stream"]):
        st["work"].copy_(st["uvwp"])
    _assemble(st, st["work"])
    s.solve(METHODS[case["method"]], fcap.STOP_L1, SOLVE_TOL, 20_000)
    s.grad_pp(2, 1, out=_address(st["dpp"]))
    _correct(st, st["work"], None)
    return {k: st[k] for k in ("dpp", "work", "flmass")}


# ------------------------------------------------------------------------------------ work

def _counts(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["mesh"] == "tets":
        n = 6 * nx * ny * nz
        return n, (4 * n - 4 * (nx * ny + ny * nz + nx * nz)) // 2
    return nx * ny * nz, (nx - 1) * ny * nz + nx * (ny - 1) * nz + nx * ny * (nz - 1)


def _iterations(case):
    """Iterations to SOLVE_TOL as measured over the boxes of this file, by their longest edge."""
    edge = max(case["nx"], case["ny"], case["nz"])
    per_edge = {"iccg": 2.7, "dpcg": 8.0, "fcg_learned": 0.7, "fcg_jacobi": 0.9}
    return max(5.0, per_edge.get(case["method"], 0.0) * edge)


def work(case):
    """Bytes and operations of one pass: matrix, factors and vectors once per iteration, each
    field and each face's geometry once per assembly; FP64 values and 32-bit indices except where
    the method keeps FP32 (flexible CG: four passes over the matrix per iteration)."""
    n, nif = _counts(case)
    nnz = 2 * nif + n
    kind, method, its = case["kind"], case["method"], _iterations(case)
    assemble = {"bytes": nif * (64 + 8) + n * (64 + 96 + 32 + 8) + 8.0 * nnz, "flops": nif * 250.0 + n * 30.0}
    if kind == "assemble":
        return assemble
    if kind == "correct":
        return {"bytes": nif * (64 + 12 + 16) + n * (8 + 24 + 32 + 24 + 64 + 16 + 8.0), "flops": nif * 100.0 + n * 30.0}
    if kind == "network_grad":
        # 4 layers, 32 channels in BF16, forward and backward; the node products and the messages
        return {"bytes": 4 * (3 * 64.0 * n + 2 * 8.0 * (nnz - n)), "flops": 3 * 4 * (4096.0 * n + 64.0 * (nnz - n))}
    if method in ("fcg_learned", "fcg_jacobi"):
        layers = 0.5 * 4 * (128 * n + 24 * n) if method == "fcg_learned" else 0.0
        its_bytes = 4 * (8.0 * nnz + 12 * n) + 120.0 * n + layers
        return {"bytes": its * its_bytes, "flops": its * (8.0 * nnz + 40 * n + (0.5 * 4 * 4352 * n if layers else 0))}
    sweeps = 0 if method == "dpcg" else 1
    per_iteration = 12.0 * nnz + sweeps * (12.0 * nnz + 24 * n) + 72.0 * n
    if kind == "momentum":
        one = 6.0 * 2 * per_iteration * (0.7 if method == "bicgstab_mixed" else 1.0)
        return {"bytes": 3 * one + 12.0 * 8 * n, "flops": 3 * 6 * 2 * (4.0 * nnz + 12 * n)}
    solve = {"bytes": its * per_iteration, "flops": its * (4.0 * nnz + 12.0 * n)}
    if kind == "simple":
        return {k: solve[k] + 1.5 * assemble[k] for k in solve}
    return solve


def tolerance(case):
    kind = case["kind"]
    if kind in ("assemble", "correct"):
        return {"rel": 1e-11, "max": 1e-9}      # FP64 sums of a handful of terms, with cancellation
    if kind == "network_grad":
        return {"rel": 1e-2}                    # BF16 activations
    return {"rel": 1e-6, "max": 1e-5}           # solved to 1e-8 of the right-hand side


# ------------------------------------------------------------------------------------ exact

class _Operator:
    """(A x)_P = sum_f c_f (x_P - x_N) + w_P x_P: with no coefficients given, the Laplacian with its
    wall terms w; else the pressure correction's matrix, which has none."""

    def __init__(self, geo, coef=None):
        n = geo.n
        wall = torch.zeros(n, dtype=torch.float64, device="cuda")
        if coef is None:
            d = geo.xc[geo.nei] - geo.xc[geo.p]
            s = geo.s[:geo.nif]
            coef = (s * s).sum(1) / (s * d).sum(1)
            cells = geo.own[geo.walls]
            wall.index_add_(0, cells, geo.s[geo.walls].norm(dim=1) / (geo.xc[cells] - geo.xf[geo.walls]).norm(dim=1))
        self.diag = wall.index_add_(0, geo.p, coef).index_add_(0, geo.nei, coef)
        rows, cols = torch.cat([geo.p, geo.nei]), torch.cat([geo.nei, geo.p])
        order = torch.argsort(rows * n + cols)
        self.rows, self.cols, self.coef = rows[order], cols[order], torch.cat([coef, coef])[order]
        ptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
        ptr[1:] = torch.cumsum(torch.bincount(rows, minlength=n), 0)
        self.off = torch.sparse_csr_tensor(ptr, self.cols, self.coef, (n, n))

    def __call__(self, x):
        return self.diag * x - self.off @ x

    def solve(self, b, tol=1e-13, most=20_000):
        x, r, p = torch.zeros_like(b), b.clone(), None
        goal, rho = tol * float(b.norm()), 1.0
        for it in range(most):
            z = r / self.diag
            rho, before = torch.dot(r, z), rho
            p = z if p is None else z + (rho / before) * p
            q = self(p)
            alpha = rho / torch.dot(p, q)
            x += alpha * p
            r -= alpha * q
            if it % 50 == 49 and float(r.norm()) <= goal:
                break
        return x


def _gradient(geo, cells, boundary):
    face = torch.cat([geo.at_faces(cells), boundary])
    g = geo.sum_faces(torch.zeros(geo.n, 3, dtype=torch.float64, device="cuda"), face[:, None] * geo.s)
    return g / geo.vol[:, None]


def _rhie_chow(geo, f, grads):
    """Coefficient and mass flux of every inner face, from the momentum-interpolation formula as the
    reference writes it (its extrapolated pressure difference subtracts the owner's x term only)."""
    s, xf = geo.s[:geo.nif], geo.xf[:geo.nif]
    xp, xn = geo.xc[geo.p], geo.xc[geo.nei]
    d, normal = xn - xp, s / s.norm(dim=1)[:, None]
    diffusivity = torch.stack([geo.at_faces(geo.vol * f["ap"][k]) for k in range(3)], 1)
    den = geo.at_faces(f["den"])
    over = 1.0 / (s * d * normal).sum(1)
    coef = den * diffusivity[:, 0] * (s * s).sum(1) * over
    value = []
    for k in range(3):
        fi, g = f["uvwp"][k, :geo.n], grads[k]
        value.append(0.5 * (fi[geo.p] + fi[geo.nei] + (g[geo.p] * (xf - xp)).sum(1) + (g[geo.nei] * (xf - xn)).sum(1)))
    p, gp = f["uvwp"][3, :geo.n], grads[3]
    project = lambda x: (xf - (xf - x) * normal) - x  # noqa: E731
    own, other = gp[geo.p] * project(xp), gp[geo.nei] * project(xn)
    dpe = p[geo.nei] - p[geo.p] + other.sum(1) - own[:, 0] + own[:, 1] + own[:, 2]
    velocity = torch.stack(value, 1) - diffusivity * (dpe * over)[:, None] * s \
        + diffusivity * geo.at_faces(gp) * d * normal
    return coef, den * (velocity * s).sum(1)


def _nonorthogonal(geo, f, gp):
    s, xf = geo.s[:geo.nif], geo.xf[:geo.nif]
    xp, xn = geo.xc[geo.p], geo.xc[geo.nei]
    are = s.norm(dim=1)
    normal = s / are[:, None]
    project = lambda x: (xf - (xf - x) * normal) - x  # noqa: E731
    rapr = geo.at_faces(f["ap"][0] * f["den"] * geo.vol)
    return rapr * are * (gp[geo.nei] * project(xn) - gp[geo.p] * project(xp)).sum(1) / ((xn - xp) * normal).sum(1)


def _exact_step(case, seed):
    geo = _Geometry(_mesh(case, seed))
    f = _step_fields(geo, seed)
    n, kind = geo.n, case["kind"]
    grads = [_gradient(geo, f["uvwp"][k, :n], f["uvwp"][k, n:]) for k in range(4)]
    coef, flux = _rhie_chow(geo, f, grads)
    zero = torch.zeros(n, dtype=torch.float64, device="cuda")
    rhs = -geo.sum_faces(zero.clone(), flux)
    op = _Operator(geo, coef)
    if kind == "assemble":
        rows = torch.cat([op.rows, torch.arange(n, device="cuda")])
        cols = torch.cat([op.cols, torch.arange(n, device="cuda")])
        a = torch.cat([-op.coef, op.diag])[torch.argsort(rows * n + cols)]
        return {"grads": torch.stack(grads).reshape(4, -1), "a": a, "rhs": rhs, "flmass": flux}
    if kind == "correct":
        pp = f["pp"][:n]
        dpp = _gradient(geo, pp, f["pp"][n:])
    else:
        pp = op.solve(rhs)
        face_cells = geo.own[geo.nif:]
        dpp = _gradient(geo, pp, pp[face_cells])
        # the second stage extrapolates to the walls with the first one's gradient
        extra = (dpp[face_cells] * (geo.xf[geo.nif:] - geo.xc[face_cells])).sum(1)
        value = torch.cat([torch.zeros(geo.nif, dtype=torch.float64, device="cuda"), pp[face_cells]])
        value[geo.walls] += extra[geo.walls.start - geo.nif:geo.walls.stop - geo.nif]
        dpp = _gradient(geo, pp, value[geo.nif:])
    flux = flux - coef * (pp[geo.nei] - pp[geo.p])
    uvwp = f["uvwp"].clone()
    for k in range(3):
        uvwp[k, :n] -= dpp[:, k] * geo.vol * f["ap"][k]
    uvwp[3, :n] += 0.3 * (pp - pp[0])
    if kind == "simple":
        return {"dpp": dpp.reshape(-1), "work": uvwp, "flmass": flux}
    more = _nonorthogonal(geo, f, dpp)
    return {"dpp": dpp.reshape(-1), "uvwp": uvwp, "flmass": flux + more, "rhs": -geo.sum_faces(zero, more)}


def _exact_momentum(case, seed):
    geo = _Geometry(_mesh(case, seed))
    flux, sp, src, phi = _momentum_inputs(geo, seed)
    s = geo.s[:geo.nif]
    de = VIS * s.norm(dim=1) / (geo.xc[geo.nei] - geo.xc[geo.p]).norm(dim=1)
    to_nei, to_own = -de + flux.clamp(max=0.0), -de - flux.clamp(min=0.0)   # coefficients of rows P and N
    total = torch.zeros(geo.n, dtype=torch.float64, device="cuda")
    total.index_add_(0, geo.p, to_nei).index_add_(0, geo.nei, to_own)
    out = {"phi": [], "ap": []}
    for c in range(3):
        diag = (sp[c] - total) / URF
        b = src[c] + (1.0 - URF) * diag * phi[c]
        x = phi[c].clone()
        # the rows' dominance makes this converge by URF a pass
        for _ in range(110):
            off = torch.zeros_like(x)
            off.index_add_(0, geo.p, to_nei * x[geo.nei]).index_add_(0, geo.nei, to_own * x[geo.p])
            x = (b - off) / diag
        out["phi"].append(x)
        out["ap"].append(1.0 / diag)
    return out


def _exact_network(case, seed):
    geo = _Geometry(_mesh(case, seed))
    op = _Operator(geo)
    r, e = (t.double() for t in _network_pair(geo, seed, op))
    d = geo.xc[op.cols] - geo.xc[op.rows]
    # face of every entry: the faces' own order is the sorted order of their (owner, neighbour) pairs
    key = geo.p * geo.n + geo.nei
    low, high = torch.minimum(op.rows, op.cols), torch.maximum(op.rows, op.cols)
    s = geo.s[:geo.nif][torch.searchsorted(key, low * geo.n + high)]
    size, dist = s.norm(dim=1), d.norm(dim=1)
    e1, e2 = size / dist / op.diag[op.rows], 1.0 - (s * d).sum(1).abs() / (size * dist)
    theta = torch.from_numpy(np.load(gnn.DEFAULT_WEIGHTS, allow_pickle=False)).cuda().double().requires_grad_()
    h_, at = gnn.H, gnn.OFF_LAYER0
    v = r / op.diag
    scale = (v * v).mean().sqrt() + 1e-30
    u = v / scale
    h = torch.relu(u[:, None] * theta[:h_] + theta[h_:2 * h_])
    for _ in range(gnn.L):
        ws, wm = theta[at:at + h_ * h_].reshape(h_, h_), theta[at + h_ * h_:at + 2 * h_ * h_].reshape(h_, h_)
        b, g = theta[at + 2 * h_ * h_:][:h_], theta[at + 2 * h_ * h_ + h_:][:3]
        message = (g[0] + g[1] * e1 + g[2] * e2)[:, None] * h[op.cols]
        agg = torch.zeros_like(h).index_add(0, op.rows, message)
        h = h + torch.relu(h @ ws.T + agg @ wm.T + b)
        at += gnn.LAYER_STRIDE
    z = scale * (u + h @ theta[gnn.OFF_DEC_W:gnn.OFF_DEC_W + h_] + theta[gnn.OFF_DEC_B])
    norm = torch.dot(e, op(e))
    diff = z - e
    (grad,) = torch.autograd.grad(z, theta, 2.0 * op(diff.detach()) / norm)
    return {"loss": float(torch.dot(diff, op(diff)) / norm), "grad": grad.detach()}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("simple", "assemble", "correct"):
        return _exact_step(case, seed)
    if kind == "momentum":
        return _exact_momentum(case, seed)
    if kind == "network_grad":
        return _exact_network(case, seed)
    geo = _Geometry(_mesh(case, seed))
    return _Operator(geo).solve(_blobs(_generator(seed), geo))

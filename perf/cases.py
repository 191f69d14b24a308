"""The work a program has this framework do: edge loops that add into shared
mesh data, over the sizes, orderings, layouts and strategies of the
repository's own configurations, and the training of the cost model.

A case names a mesh, how its loop is planned and what one pass is: one step
("iters" 0, as a time loop calls it) or one call of `run` with that many
iterations (with the copies in and out that the reference's loops make).
The mesh, its ordering and its partition are fixed by the case; the fields on
it come from the seed.  The buffers are torch tensors on the GPU, handed to the
loop by address.
"""
import math

import numpy as np
import torch

from cuda_fot_amd import Problem, capi, mini_aero_problem, meshgen, res_calc_problem, volna_problem
from cuda_fot_amd.device import Batch, Loop
from cuda_fot_amd.mlp import MLP

DEVICE = "cuda"


def listed():
    return [
        # a mesh of a few thousand edges: launches and latency are all there is
        dict(name="airfoil tiny", kind="airfoil", nx=64, ny=32, plan="owner", block=240, soa=False, iters=0),
        # the headline loop and size: owner compute on a renumbered mesh
        dict(name="airfoil", kind="airfoil", nx=1200, ny=600, plan="owner", block=240, soa=False, iters=0),
        # the same beyond the last-level cache
        dict(name="airfoil large", kind="airfoil", nx=2400, ny=1200, plan="owner", block=240, soa=False, iters=0),
        # the reference's own plan: one launch per block colour, SOA, a whole
        # loop call of several iterations, ragged sizes
        dict(name="airfoil colours", kind="airfoil", nx=701, ny=463, plan="colours", block=512, soa=True, iters=10),
        # the plan-free loop: FP64 atomics on a bandwidth-ordered mesh
        dict(name="airfoil atomics", kind="airfoil", nx=1200, ny=600, plan="atomics", block=256, soa=False, iters=0),
        # the synthetic increment, whose iterate is copied back every iteration
        dict(name="mine", kind="mine", nx=1024, ny=1024, block=512, soa=False, iters=10),
        # 3D element corner scatter, ragged sizes, beyond the last-level cache
        dict(name="hex", kind="hex", nx=103, ny=110, nz=97, block=512, soa=False, iters=0),
        # 3D face flux: much FP64 arithmetic and wide gathered rows
        dict(name="mini_aero", kind="mini_aero", nx=80, ny=80, nz=80, block=128, soa=False, iters=0),
        # 3D element forces and the element volume, one whole call
        dict(name="lulesh", kind="lulesh", nx=96, ny=96, nz=96, block=512, soa=False, iters=1),
        # 2D corner scatter, many cell arrays
        dict(name="getacc", kind="getacc", nx=1024, ny=1024, block=512, soa=False, iters=0),
        # many uneven triangle meshes in one launch
        dict(name="volna batch", kind="volna", meshes=32, low=10000, high=200000, block=512, soa=False, iters=0),
        # the cost model's training on the tuner's corpus (rows x features)
        dict(name="cost model", kind="mlp", rows=695, epochs=20),
    ]


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["airfoil", "airfoil", "airfoil", "mine", "hex", "mini_aero", "lulesh", "getacc", "volna", "mlp"])
    soa = rng.random() < 0.3
    if kind == "mlp":
        return dict(kind=kind, rows=_spread(rng, 64, 2048), epochs=rng.randint(4, 20))
    if kind == "volna":
        low = _spread(rng, 2000, 20000)
        return dict(kind=kind, meshes=rng.randint(3, 24), low=low, high=low * rng.randint(2, 8), block=rng.choice([256, 512]),
                    soa=soa, iters=rng.choice([0, 0, 3]))
    if kind == "airfoil":
        plan = rng.choice(["owner", "owner", "colours", "atomics"])
        nx = _spread(rng, 40, 1500)
        return dict(kind=kind, nx=nx, ny=max(8, int(nx * rng.uniform(0.3, 1.0))), plan=plan,
                    block={"owner": 240, "colours": rng.choice([256, 512, 1024]), "atomics": 256}[plan], soa=soa,
                    iters=rng.choice([0, 0, 4]))
    if kind in ("mine", "getacc"):
        nx = _spread(rng, 48, 1000)
        return dict(kind=kind, nx=nx, ny=max(16, int(nx * rng.uniform(0.4, 1.0))), block=rng.choice([256, 512]), soa=soa,
                    iters=rng.randint(2, 8) if kind == "mine" else 0)
    top = {"hex": 96, "mini_aero": 76, "lulesh": 90}[kind]
    nx, ny, nz = (rng.randint(10, top) for _ in range(3))
    return dict(kind=kind, nx=nx, ny=ny, nz=nz, block=rng.choice([128, 256]) if kind == "mini_aero" else rng.choice([256, 512]),
                soa=soa, iters=1 if kind == "lulesh" else 0)


# ---- meshes: fixed by the case, made once per process ---------------------


def _bisect(coords, block):
    """Recursive coordinate bisection into equal parts of at most `block`
    cells: a part id per cell."""
    n, dim = coords.shape
    part = np.empty(n, np.uint32)
    span = int(coords.max()) + 1
    c = coords.astype(np.int64)
    todo = [(np.arange(n), 0, -(-n // block))]
    while todo:
        ids, first, parts = todo.pop()
        if parts == 1:
            part[ids] = first
            continue
        here = c[ids]
        key = np.zeros(len(ids), np.int64)
        for a in np.argsort(here.min(0) - here.max(0), kind="stable"):
            key = key * span + here[:, a]
        left = parts // 2
        at = len(ids) * left // parts
        order = np.argpartition(key, at)
        todo.append((ids[order[:at]], first, left))
        todo.append((ids[order[at:]], first + left, parts - left))
    return part


def _blocks(p, coords, block):
    """The problem on compact blocks: cells sorted by part, points renumbered."""
    p.partition_vector = _bisect(coords, block)
    p.reorder_to_partition()
    p.renumber_points()
    return p


def _mesh(case):
    kind, soa = case["kind"], case["soa"]
    if kind == "airfoil":
        p = res_calc_problem(meshgen.airfoil(case["nx"], case["ny"], seed=0, shuffle=7), case["block"], soa)
        if case["plan"] == "owner":
            p.partition_points(case["block"])
        else:
            p.reorder("gps")
        return p
    if kind == "volna":
        rng, found = np.random.default_rng(0), []
        for i in range(case["meshes"]):
            cells = math.exp(rng.uniform(math.log(case["low"]), math.log(case["high"])))
            nx = max(4, int(round(math.sqrt(cells / 2 * rng.uniform(0.5, 2.0)))))
            p = volna_problem(meshgen.tri_mesh(nx, max(4, int(round(cells / 2 / nx))), seed=100 + i), case["block"], soa)
            p.partition_points(case["block"])
            found.append(p)
        return found
    if kind == "mine":
        n, m = case["nx"], case["ny"]
        edges = meshgen.grid_edges(n, m)
        at = edges.astype(np.int64).min(1)
        return _blocks(Problem([edges], [n * m], [None], [], case["block"], soa), np.stack([at // m, at % m], 1), case["block"])
    if kind == "getacc":
        n, m = case["nx"] + 1, case["ny"] + 1
        cells = meshgen.quad_grid(n, m)
        cells = cells[meshgen.permutation(cells.shape[0], 1)]
        at = cells.astype(np.int64).min(1)
        return _blocks(Problem([cells], [n * m], [None], [], case["block"], soa), np.stack([at // m, at % m], 1), case["block"])
    if kind == "mini_aero":
        p = mini_aero_problem(meshgen.hex_faces(case["nx"], case["ny"], case["nz"], seed=0), case["block"], soa)
        centre = (p.cell_data[0][:3] * 2).round().astype(np.int64).T
        return _blocks(p, centre, case["block"])
    n1, n2, n3 = case["nx"] + 1, case["ny"] + 1, case["nz"] + 1
    cells = meshgen.hex_grid(n1, n2, n3)
    cells = cells[meshgen.permutation(cells.shape[0], 1)]
    points = np.arange(n1 * n2 * n3)
    lattice = np.stack([points // n2 % n1, points % n2, points // (n1 * n2)], 1)
    at = lattice[cells.astype(np.int64)].min(1)
    xyz = lattice.astype(np.float64)
    maps, data = ([cells, cells], [None, xyz.T.copy() if soa else xyz]) if kind == "lulesh" else ([cells], [None])
    return _blocks(Problem(maps, [points.size] * len(maps), data, [], case["block"], soa), at, case["block"])


_meshes = {}


def _mesh_of(case):
    key = tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "iters")))
    if key not in _meshes:
        _meshes[key] = _mesh(case)
    return _meshes[key]


# ---- the fields on them, from the seed -------------------------------------


class _Fields:
    """Seeded FP64 tensors on the GPU, point data in the case's layout."""

    def __init__(self, seed, soa):
        self.gen, self.soa = torch.Generator(device=DEVICE).manual_seed(seed), soa

    def uniform(self, *shape, low=0.0, high=1.0):
        return torch.rand(shape, generator=self.gen, device=DEVICE, dtype=torch.float64) * (high - low) + low

    def normal(self, *shape, sd=1.0):
        return torch.randn(shape, generator=self.gen, device=DEVICE, dtype=torch.float64) * sd

    def points(self, t):
        """(points, dim) in the layout the loop takes."""
        return t.T.contiguous() if self.soa else t.contiguous()


def _up(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEVICE)


def _airfoil_fields(p, f):
    nc = p.num_points[0]
    free = torch.tensor([1.0, 0.4, 0.0, 2.5], dtype=torch.float64, device=DEVICE)
    q = free * (1 + 1e-2 * f.normal(nc, 4))
    return [f.points(f.normal(nc, 4, sd=0.1)), _up(p.point_data[1]), f.points(q), f.uniform(nc, low=0.5, high=1.5)], []


def _mine_fields(p, f):
    return [f.points(f.uniform(p.num_points[0], 4))], [f.uniform(4, p.num_cells)]


def _hex_fields(p, f):
    return [f.points(f.normal(p.num_points[0], 3))], [f.normal(24, p.num_cells)]


def _mini_aero_fields(p, f):
    nc = p.num_points[0]
    free = torch.tensor([1.0, 50.0, 10.0, 5.0, 216600.0], dtype=torch.float64, device=DEVICE)
    fixed = p.point_data[1][5:8].T if f.soa else p.point_data[1][:, 5:8]
    cells = torch.cat([free * (1 + 1e-2 * f.normal(nc, 5)), _up(fixed), f.normal(nc, 15, sd=1e-3), f.uniform(nc, 5)], 1)
    return [f.points(f.normal(nc, 5)), f.points(cells)], [_up(p.cell_data[0])]


def _lulesh_fields(p, f):
    xyz = _up(p.point_data[1])
    xyz = xyz + f.uniform(*xyz.shape, low=-0.2, high=0.2)
    return [f.points(f.normal(p.num_points[0], 3)), xyz], [f.normal(3, p.num_cells), f.uniform(1, p.num_cells)]


def _getacc_fields(p, f):
    nc = p.num_cells
    mass = f.uniform(4, nc) * (f.uniform(4, nc) >= 1 / 3)
    return ([f.points(f.uniform(p.num_points[0], 4))],
            [mass, f.uniform(1, nc, low=0.5, high=1.5), f.uniform(4, nc), f.normal(4, nc), f.normal(4, nc)])


def _volna_fields(p, f):
    nc, ne = p.num_points[0], p.num_cells
    state = torch.cat([f.uniform(nc, 1, low=0.5, high=2.0), f.normal(nc, 2, sd=0.1), f.uniform(nc, 1, low=-1.0, high=0.0)], 1)
    return ([f.points(state), _up(p.point_data[1])],
            [f.normal(3, ne, sd=0.1), f.normal(2, ne, sd=0.1), _up(p.cell_data[2]), _up(p.cell_data[3])])


_FIELDS = dict(airfoil=_airfoil_fields, mine=_mine_fields, hex=_hex_fields, mini_aero=_mini_aero_fields,
               lulesh=_lulesh_fields, getacc=_getacc_fields, volna=_volna_fields)


def _mlp_inputs(case, seed):
    """Standardised features and log times as the tuner gives them, a mask
    with some classes unmeasured, He-uniform weights."""
    g = np.random.default_rng(seed)
    rows, sizes = case["rows"], (24, 64, 64, 6)
    x = g.standard_normal((rows, 24)).astype(np.float32)
    mix = g.standard_normal((24, 6)) / 5
    t = (np.tanh(x @ mix) + 0.1 * g.standard_normal((rows, 6))).astype(np.float32)
    mask = (g.random((rows, 6)) < 0.9).astype(np.float32)
    params = []
    for i, o in zip(sizes, sizes[1:]):
        a = math.sqrt(6.0 / i)
        params += [g.uniform(-a, a, i * o), np.zeros(o)]
    return x, t, mask, np.concatenate(params).astype(np.float32)


# ---- preparing and running -------------------------------------------------


class _Buffer:
    """A tensor as the loop takes it: address and shape."""

    def __init__(self, t):
        self.tensor, self.ptr, self.shape = t, t.data_ptr(), tuple(t.shape)


def _functor(kind):
    return {"airfoil": lambda: capi.functor(capi.KERNEL_RES_CALC), "mine": lambda: capi.functor(capi.KERNEL_MINE, 2, 4, 4),
            "hex": lambda: capi.functor(capi.KERNEL_HEX_SCATTER), "mini_aero": lambda: capi.functor(capi.KERNEL_MINI_AERO),
            "lulesh": lambda: capi.functor(capi.KERNEL_LULESH), "getacc": lambda: capi.functor(capi.KERNEL_GETACC),
            "volna": lambda: capi.functor(capi.KERNEL_VOLNA)}[kind]()


def _buffers(p, case, f):
    points, cells = _FIELDS[case["kind"]](p, f)
    return [_Buffer(t) for t in points], _Buffer(points[0].clone()), [_Buffer(t) for t in cells]


def prepare(case, seed):
    if case["kind"] == "mlp":
        x, t, mask, params = _mlp_inputs(case, seed)
        net = MLP(24, 64, 6)
        net.set_params(params)
        return dict(case=case, net=net, x=x, t=t, mask=mask)
    f, mesh = _Fields(seed, case["soa"]), _mesh_of(case)
    if case["kind"] == "volna":
        parts = [_buffers(p, case, f) for p in mesh]
        torch.cuda.synchronize()
        loop = Batch(_functor("volna"), [dict(maps=p.maps, num_points=p.num_points, point_data=pd, out=out, cell_data=cd, soa=case["soa"],
                                              block_size=case["block"], point_partition=p.point_partition)
                                         for p, (pd, out, cd) in zip(mesh, parts)])
        return dict(case=case, loop=loop, results=[(pd[0] if case["iters"] else out).tensor for pd, out, _ in parts], keep=parts)
    points, out, cells = _buffers(mesh, case, f)
    torch.cuda.synchronize()
    strategy, partition, flags = capi.STRATEGY_HIERARCHICAL, mesh.partition_vector, capi.LOOP_TWO_PHASE
    if case["kind"] == "airfoil" and case["plan"] == "owner":
        partition = mesh.point_partition
        flags = capi.LOOP_OWNER_COMPUTE | capi.LOOP_POINT_PARTITION | capi.LOOP_TWO_PER_THREAD | capi.LOOP_OWNER_GATHER
    elif case["kind"] == "airfoil":
        flags = capi.LOOP_STAGE_INPUTS if case["plan"] == "colours" else 0
        strategy = strategy if case["plan"] == "colours" else capi.STRATEGY_ATOMIC
    loop = Loop(_functor(case["kind"]), mesh.maps, mesh.num_points, points, out, cells, soa=case["soa"], strategy=strategy,
                block_size=case["block"], partition=partition, flags=flags)
    results = [(points[0] if case["iters"] else out).tensor]
    if case["kind"] == "lulesh":
        results.append(cells[1].tensor)  # the element volumes
    return dict(case=case, loop=loop, results=results, keep=(points, out, cells))


def run(state):
    case = state["case"]
    if case["kind"] == "mlp":
        losses = state["net"].train(state["x"], state["t"], state["mask"], epochs=case["epochs"], lr=3e-3, weight_decay=1e-4)
        return dict(losses=losses, params=state["net"].get_params())
    if case["iters"]:
        state["loop"].run(case["iters"])
    else:
        state["loop"].step()
    return state["results"]


# ---- what a pass cannot do without -----------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        params, rows = 24 * 64 + 64 * 64 + 64 * 6 + 134, case["rows"]
        return dict(bytes=case["epochs"] * 4 * (36 * rows + 6 * params), flops=case["epochs"] * 6 * params * rows)
    times = max(1, case["iters"])
    if kind == "volna":
        cells = sum(p.num_points[0] for p in _mesh_of(case))
        edges = sum(p.num_cells for p in _mesh_of(case))
        return dict(bytes=times * 72 * (cells + edges), flops=times * 25 * edges)
    x, y, z = case["nx"], case["ny"], case.get("nz", 0)
    if kind == "airfoil":
        cells, nodes, edges = x * y, (x + 1) * (y + 1), x * (y - 1) + (x - 1) * y
        b, fl = 16 * nodes + 104 * cells + 16 * edges, 75 * edges
    elif kind == "mine":
        edges = x * (y - 1) + (x - 1) * y
        b, fl = 96 * x * y + 40 * edges, 24 * edges
    elif kind == "getacc":
        b, fl = 64 * (x + 1) * (y + 1) + 152 * x * y, 32 * x * y
    elif kind == "hex":
        b, fl = 48 * (x + 1) * (y + 1) * (z + 1) + 224 * x * y * z, 24 * x * y * z
    elif kind == "lulesh":
        b, fl = 72 * (x + 1) * (y + 1) * (z + 1) + 64 * x * y * z, 400 * x * y * z
    else:
        faces = (x - 1) * y * z + x * (y - 1) * z + x * y * (z - 1)
        b, fl = 304 * x * y * z + 104 * faces, 1000 * faces
    return dict(bytes=times * b, flops=times * fl)


# ---- the same in plain torch, 64 bits --------------------------------------


def _airfoil_increments(m, pd, cd):
    x, q, adt = pd[1], pd[2], pd[3]
    a, b = m[0].T
    dx, dy = (x[m[1][:, 0]] - x[m[1][:, 1]]).T

    def side(c):
        r, u, v, e = q[c].T
        return 0.4 * (e - 0.5 * (u * u + v * v) / r), (u * dy - v * dx) / r

    (p1, v1), (p2, v2) = side(a), side(b)
    mu = 0.5 * (adt[a] + adt[b]) * 0.05
    q1, q2 = q[a].T, q[b].T
    flux = [0.5 * (v1 * q1[0] + v2 * q2[0]), 0.5 * (v1 * q1[1] + p1 * dy + v2 * q2[1] + p2 * dy),
            0.5 * (v1 * q1[2] - p1 * dx + v2 * q2[2] - p2 * dx), 0.5 * (v1 * (q1[3] + p1) + v2 * (q2[3] + p2))]
    flux = torch.stack([fl + mu * (q1[d] - q2[d]) for d, fl in enumerate(flux)], 1)
    return torch.stack([flux, -flux], 1)


def _mine_increments(m, pd, cd):
    w = cd[0].T
    return torch.stack([2 * pd[0][m[0][:, 1]] * w, 2 * pd[0][m[0][:, 0]] * w], 1)


def _hex_increments(m, pd, cd):
    return cd[0].reshape(3, 8, -1).permute(2, 1, 0)


def _getacc_increments(m, pd, cd):
    mass, rho, wt, fx, fy = cd
    before = mass.roll(1, 0)
    first = torch.where(mass > 1e-40, mass, torch.where(before > 1e-40, before, rho * wt))
    return torch.stack([first, wt, fx, fy], 0).permute(2, 1, 0)


def _lulesh_increments(m, pd, cd):
    c = pd[1][m[0]]  # (elements, 8, 3)
    faces = [(0, 1, 2, 3), (0, 4, 5, 1), (1, 5, 6, 2), (2, 6, 7, 3), (3, 7, 4, 0), (4, 7, 6, 5)]
    normal = torch.zeros_like(c)
    for a, b, e, d in faces:
        s = 0.5 * (c[:, d] + c[:, e] - c[:, b] - c[:, a])
        t = 0.5 * (c[:, e] + c[:, b] - c[:, d] - c[:, a])
        area = 0.25 * torch.linalg.cross(s, t)
        for k in (a, b, e, d):
            normal[:, k] += area
    return -cd[0].T[:, None, :] * normal


def _lulesh_volume(m, pd):
    c = pd[1][m[0]]
    d = [c[:, 6] - c[:, 0], c[:, 5] - c[:, 3], c[:, 7] - c[:, 1], c[:, 4] - c[:, 2]]
    xi, et, ze = (0.125 * (d[0] + s * d[1] + t * d[2] + u * d[3]) for s, t, u in ((1, -1, -1), (-1, 1, -1), (1, 1, 1)))
    return 8 * (et * torch.linalg.cross(ze, xi)).sum(1)


def _volna_increments(m, pd, cd):
    flux, bathy, normal, boundary = cd
    v0, v1 = pd[1][m[0][:, 0]], pd[1][m[0][:, 1]]
    inside = (boundary[0] == 0).double()
    sides = []
    for k, v in ((0, -1 / v0), (1, inside / v1)):
        sides.append(torch.stack([flux[0] * v, (flux[1] + bathy[k] * normal[0]) * v, (flux[2] + bathy[k] * normal[1]) * v, 0 * v], 1))
    return torch.stack(sides, 1)


def _mini_aero_increments(m, pd, cd):
    at, n, t, b = (cd[0][3 * k:3 * k + 3].T for k in range(4))

    def side(c):
        v = pd[1][c]
        r = v[:, 0]
        vel = v[:, 1:4] / r[:, None]
        temp = (v[:, 4] / r - 0.5 * (vel * vel).sum(1)) * 0.4 / 287.05
        grad = v[:, 8:23].reshape(-1, 5, 3)
        prim = torch.cat([r[:, None], vel, temp[:, None]], 1)
        return prim + (grad * (at - v[:, 5:8])[:, None, :]).sum(2) * v[:, 23:28], grad

    (pl, gl), (pr, gr) = side(m[0][:, 0]), side(m[0][:, 1])

    def state(p):
        r, vel, temp = p[:, 0], p[:, 1:4], p[:, 4]
        pres, h = r * 287.05 * temp, 1004.0 * temp
        return r, vel, pres, h, h + 0.5 * (vel * vel).sum(1), r * (n * vel).sum(1)

    rl, ul, prl, hl, Hl, ml = state(pl)
    rr, ur, prr, hr, Hr, mr = state(pr)
    mom = 0.5 * (ml[:, None] * ul + mr[:, None] * ur + n * (prl + prr)[:, None])
    flux = torch.cat([(0.5 * (ml + mr))[:, None], mom, (0.5 * (ml * Hl + mr * Hr))[:, None]], 1)
    nn = n.norm(dim=1)
    nu, tu, bu = n / nn[:, None], t / t.norm(dim=1)[:, None], b / b.norm(dim=1)[:, None]
    al = rl.sqrt() / (rl.sqrt() + rr.sqrt())
    be = 1 - al
    vel = al[:, None] * ul + be[:, None] * ur
    h = al * hl + be * hr + 0.5 * al * be * ((ur - ul) ** 2).sum(1)
    c = (0.4 * h).sqrt()
    vn, vt, vb = (vel * nu).sum(1), (vel * tu).sum(1), (vel * bu).sum(1)
    ke = 0.5 * (vel * vel).sum(1)
    dm = rr[:, None] * ur - rl[:, None] * ul
    de = (rr * Hr - prr) - (rl * Hl - prl)
    dr = rr - rl
    cbar, ubar = c * nn, (vel * n).sum(1)
    eps = 0.1 * (ubar.abs() + cbar)

    def fixed(e):
        return torch.where(e.abs() < eps, 0.5 * (e * e + eps * eps) / eps, e.abs())

    e1, e2, e3 = fixed(ubar + cbar), fixed(ubar - cbar), fixed(ubar)
    kh, he = ke - h, h + ke
    dot = (vel * dm).sum(1)
    l1 = e1 * ((0.4 * kh + c * (c - vn)) * dr + c * (nu * dm).sum(1) - 0.4 * dot + 0.4 * de)
    l2 = e2 * ((0.4 * kh + c * (c + vn)) * dr - c * (nu * dm).sum(1) - 0.4 * dot + 0.4 * de)
    l3 = e3 * (kh * dr - dot + de)
    l4 = e3 * (-vt * dr + (tu * dm).sum(1))
    l5 = e3 * (-vb * dr + (bu * dm).sum(1))
    i = 1 / (c * c)
    rows = [0.5 * i * (l1 + l2) - 0.4 * i * l3]
    for k in range(3):
        rows.append(0.5 * i * ((vel[:, k] + nu[:, k] * c) * l1 + (vel[:, k] - nu[:, k] * c) * l2) - 0.4 * i * vel[:, k] * l3
                    + tu[:, k] * l4 + bu[:, k] * l5)
    rows.append(0.5 * i * ((he + c * vn) * l1 + (he - c * vn) * l2) + (c * c - 0.4 * he) * i * l3 + vt * l4 + vb * l5)
    flux = flux - 0.5 * torch.stack(rows, 1)
    mid, grad = 0.5 * (pl + pr), 0.5 * (gl + gr)
    temp = mid[:, 4]
    mu = 1.458e-6 * temp * temp.sqrt() / (temp + 110.4)
    g = grad[:, 1:4]
    strain = 0.5 * (g + g.transpose(1, 2))
    strain = strain - (g.diagonal(dim1=1, dim2=2).sum(1) / 3)[:, None, None] * torch.eye(3, dtype=torch.float64, device=DEVICE)
    stress = (2 * mu[:, None, None] * strain * n[:, None, :]).sum(2)
    heat = (mu * 1006.0 / 0.71) * (grad[:, 4] * n).sum(1)
    flux = flux - torch.cat([torch.zeros_like(heat)[:, None], stress, ((stress * mid[:, 1:4]).sum(1) + heat)[:, None]], 1)
    return torch.stack([-flux, flux], 1)


_INCREMENTS = dict(airfoil=_airfoil_increments, mine=_mine_increments, hex=_hex_increments, mini_aero=_mini_aero_increments,
                   lulesh=_lulesh_increments, getacc=_getacc_increments, volna=_volna_increments)


def _loop_exact(p, case, f):
    points, cells = _FIELDS[case["kind"]](p, f)
    soa = case["soa"]
    pd = [t.T.contiguous() if soa and t.dim() > 1 else t for t in points]
    m = [_up(k.astype(np.int64)) for k in p.maps]
    value = pd[0]
    for i in range(max(1, case["iters"])):
        if i == 0 or case["kind"] == "mine":
            inc = _INCREMENTS[case["kind"]](m, [value] + pd[1:], cells)
        value = value.index_add(0, m[0].reshape(-1), inc.reshape(-1, inc.shape[2]))
    found = [value.T.contiguous() if soa else value]
    if case["kind"] == "lulesh":
        found.append(_lulesh_volume(m, pd)[None])
    return found


def _mlp_exact(case, seed):
    x, t, mask, params = (torch.from_numpy(a).double() for a in _mlp_inputs(case, seed))
    params.requires_grad_(True)
    m, v, losses = torch.zeros_like(params), torch.zeros_like(params), []
    shapes = [(64, 24), (64,), (64, 64), (64,), (6, 64), (6,)]
    b1, b2 = float(np.float32(0.9)), float(np.float32(0.999))
    eps, lr, decay = float(np.float32(1e-8)), float(np.float32(3e-3)), float(np.float32(1e-4))
    for step in range(1, case["epochs"] + 1):
        w = [s.reshape(k) for s, k in zip(params.split([math.prod(k) for k in shapes]), shapes)]
        h = torch.relu(torch.relu(x @ w[0].T + w[1]) @ w[2].T + w[3])
        loss = (mask * (h @ w[4].T + w[5] - t) ** 2).sum() / mask.sum()
        grad, = torch.autograd.grad(loss, params)
        losses.append(float(loss))
        with torch.no_grad():
            g = grad + decay * params
            m, v = b1 * m + (1 - b1) * g, b2 * v + (1 - b2) * g * g
            rate = lr * math.sqrt(1 - b2 ** step) / (1 - b1 ** step)
            params = params - rate * m / (v.sqrt() + eps)
        params.requires_grad_(True)
    return dict(losses=np.array(losses), params=params.detach().numpy())


def exact(case, seed):
    if case["kind"] == "mlp":
        return _mlp_exact(case, seed)
    f, mesh = _Fields(seed, case["soa"]), _mesh_of(case)
    if case["kind"] == "volna":
        return [_loop_exact(p, case, f)[0] for p in mesh]
    return _loop_exact(mesh, case, f)

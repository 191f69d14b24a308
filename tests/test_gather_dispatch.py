"""Which hierarchical plans gather their sums, and that either kernel gives the
oracle's bits.  The rule is restated here on the host plan; the loop's LDS size
tells which kernel was planned."""
import copy

import numpy as np
import pytest

import oracle as O
from cuda_fot_amd import (Problem, capi, getacc_problem, lulesh_problem, meshgen,
                          mini_aero_problem, plan, volna_problem)
from helpers import (airfoil_problem, assert_bitwise, assert_close_scaled, hex_problem,
                     mine_problem, oracle_of)

TP = capi.LOOP_TWO_PHASE
STAGED_DIM = {O.MINI_AERO: 28, O.LULESH: 3}


def host_plan(p, block_size):
    """Per-block increments per cached point (the mean of the plan), the longest
    list, the most cached points and the workgroup's threads."""
    md, cached, most, longest, cells, blocks = p.maps[0].shape[1], 0, 0, 0, 0, 0
    for c in plan.hplan(p.maps, p.num_points[0], block_size, p.partition_vector):
        off, ids = c["block_offsets"], c["cell_list"][0].reshape(md, -1)
        for b in range(len(off) - 1):
            n = np.bincount(ids[:, off[b]:off[b + 1]].ravel())
            cached, most, longest = cached + n.size, max(most, n.size), max(longest, n.max())
            cells, blocks = max(cells, off[b + 1] - off[b]), blocks + 1
    threads = max(64, -(-int(cells) // 64) * 64)
    return dict(per_point=p.maps[0].size / cached, longest=int(longest), most=int(most),
                threads=threads, blocks=blocks)


def gathers(p, kernel, h, two_phase):
    md, td = p.maps[0].shape[1], p.point_data[0].shape[0 if p.soa else 1]
    if h["longest"] > 8 or h["most"] > 2 * h["threads"]:
        return False
    if md == 2:
        if p.soa:
            low = 2.5 if kernel in STAGED_DIM else 1.6
            return not (two_phase and h["blocks"] > 1024 and h["per_point"] < low)
        return h["per_point"] >= 2.4
    return True


def lds_of(p, kernel, h, gather):
    md, td = p.maps[0].shape[1], p.point_data[0].shape[0 if p.soa else 1]
    if not gather:
        return 8 * td * h["most"]
    dims = td if md == 2 and td <= 5 else 1 if md >= 8 else 8 // md
    planes = 8 * min(dims, td) * (md * h["threads"] + 1)
    staged = STAGED_DIM.get(kernel, 0)
    return max(planes, 8 * (staged | 1) * h["most"] if staged else 0)


def check(p, kernel, functor, block_size, iters, expect, flags=(0, TP)):
    """Runs the loop per colour and two-phase against the oracle's replay, on
    the kernel expected (a bool, or one per entry of flags)."""
    h = host_plan(p, block_size)
    o = oracle_of(p, kernel)
    o.loop_hier_replay(O.OraclePlan(p.maps, p.num_points[0], block_size, p.partition_vector), iters)
    start = [None if d is None else d.copy() for d in p.point_data]
    for k, f in enumerate(flags):
        want = expect if isinstance(expect, bool) else expect[k]
        assert gathers(p, kernel, h, f & TP) == want, h
        p.point_data = [None if d is None else d.copy() for d in start]
        stats = p.gpu_loop(functor, capi.STRATEGY_HIERARCHICAL, iters, block_size=block_size, flags=f)
        assert stats["lds_bytes"] == lds_of(p, kernel, h, want), (f, h, stats)
        assert_bitwise(p.point_data[0], o.target, f"flags {f} {h}")
    return h


@pytest.mark.gpu
@pytest.mark.parametrize("soa", [False, True])
@pytest.mark.parametrize("kind,block_size,gather", [("airfoil", 128, False), ("airfoil", 256, True),
                                                    ("mine", 128, False), ("mine", 256, True),
                                                    ("volna", 128, False), ("volna", 512, True),
                                                    ("mini_aero", 128, False),
                                                    ("mini_aero", 512, True)])
def test_two_point_cells_gather_where_points_add_enough(gpu, kind, block_size, gather, soa):
    """GPS-ordered meshes on either side of 2.4 increments per cached point: AOS
    plans below keep the colour loop, SOA plans gather."""
    if kind == "airfoil":
        p, kernel, f = airfoil_problem(160, 80, soa=soa, res0_seed=3), O.RES_CALC, capi.KERNEL_RES_CALC
    elif kind == "mine":
        p, kernel, f = mine_problem(160, 80, soa=soa), O.MINE2, None
    elif kind == "volna":
        p, kernel, f = volna_problem(meshgen.tri_mesh(80, 80, seed=1), soa=soa), O.VOLNA, capi.KERNEL_VOLNA
    else:
        p, kernel, f = mini_aero_problem(meshgen.hex_faces(34, 34, 34), soa=soa), O.MINI_AERO, \
            capi.KERNEL_MINI_AERO
    p.reorder("gps")
    f = capi.functor(capi.KERNEL_MINE, 2, 4, 4) if f is None else capi.functor(f)
    check(p, kernel, f, block_size, 2 if kind == "mine" else 1, gather or soa)


@pytest.mark.gpu
def test_large_soa_plans_of_few_increments_per_point(gpu):
    p = volna_problem(meshgen.tri_mesh(220, 220, seed=1), soa=True)
    p.reorder("gps")
    h = check(p, O.VOLNA, capi.functor(capi.KERNEL_VOLNA), 128, 1, (True, False))
    assert h["blocks"] > 1024 and h["per_point"] < 1.6
    p = volna_problem(meshgen.tri_mesh(120, 120, seed=1), soa=True)
    p.reorder("gps")
    h = check(p, O.VOLNA, capi.functor(capi.KERNEL_VOLNA), 128, 1, True)
    assert h["blocks"] <= 1024
    p = mini_aero_problem(meshgen.hex_faces(36, 36, 36), soa=True)
    p.reorder("gps")
    h = check(p, O.MINI_AERO, capi.functor(capi.KERNEL_MINI_AERO), 128, 1, (True, False))
    assert h["blocks"] > 1024 and 2.0 < h["per_point"] < 2.5


# ---- owner compute -----------------------------------------------------------
def owner_lds(p, op, gather):
    """LDS of the loop of its own on this plan (gathered sums or colour loop)."""
    md, td = p.maps[0].shape[1], p.point_data[0].shape[0 if p.soa else 1]
    if not gather:
        return (8 * td + 4) * int(op["blk_owned"].max())
    cap = int(np.diff(op["blk_cell_off"]).max())
    return 8 * (min(td, 2) if md == 2 else 1) * (md * cap + 1)


def owner_gathers(p, kernel, op):
    md, cells, owned = p.maps[0].shape[1], np.diff(op["blk_cell_off"]), op["blk_owned"]
    threads = max(64, -(-int(cells.max()) // 64) * 64)
    half = max(64, -(-max(-(-int(cells.max()) // 2), int(owned.max())) // 64) * 64)
    consecutive = all(np.all(np.diff(op["cached"][c:c + n].astype(np.int64)) == 1)
                      for c, n in zip(op["blk_cache_off"], owned))
    scattered = kernel == O.GETACC or (kernel == O.MINE2 and not p.soa and
                                       op["cells"].size >= 1 << 18)
    return 4 * half <= 3 * threads and (consecutive or scattered)


@pytest.mark.gpu
@pytest.mark.parametrize("soa", [False, True])
@pytest.mark.parametrize("kind,parts,gather", [
    ("mine", "points", True), ("mine", "gps", False), ("mine large", "gps", None),
    ("volna", "points", True), ("volna", "gps", False), ("getacc", "points", True),
    ("getacc", "gps", True), ("mine4", "points", True), ("mine4", "gps", False),
    ("mine4", "kway", False), ("getacc", "kway", False)])
def test_owner_blocks_gather_where_it_is_faster(gpu, kind, parts, gather, soa):
    """Owner-compute loops on parts with consecutive ids, on GPS-ordered meshes
    and on k-way cell parts: the kernel planned, and the replay's bits."""
    md, bs = (4 if kind in ("mine4", "getacc") else 2), 256
    if kind == "volna":
        p, kernel = volna_problem(meshgen.tri_mesh(40, 33, seed=1), soa=soa), O.VOLNA
        f = capi.functor(capi.KERNEL_VOLNA)
    elif kind == "getacc":
        p, kernel, f = getacc_problem(61, 83, soa=soa), O.GETACC, capi.functor(capi.KERNEL_GETACC)
    elif kind == "mine4":
        cells = meshgen.quad_grid(70, 66)
        n = 70 * 66
        pd = meshgen.uniform(4 * n, 1).reshape(n, 4)
        p = Problem([cells[meshgen.permutation(cells.shape[0], 3)]], [n],
                    [pd.T.copy() if soa else pd], [meshgen.uniform(4 * cells.shape[0], 2).reshape(4, -1)],
                    bs, soa)
        kernel, f = O.MINE4, capi.functor(capi.KERNEL_MINE, 4, 4, 4)
    else:
        p = mine_problem(420, 330, soa=soa) if "large" in kind else mine_problem(70, 66, soa=soa)
        kernel, f = O.MINE2, capi.functor(capi.KERNEL_MINE, 2, 4, 4)
    p.block_size = bs
    part = point_part = None
    if parts == "points":
        p.partition_points(bs)
        point_part = p.point_partition
    elif parts == "gps":
        p.reorder("gps")
    else:
        p.partition(method="kway")
        p.reorder_to_partition()
        p.renumber_points()
        part = p.partition_vector
    op = plan.owner_plan(p.maps[0], p.num_points[0], bs, part, point_part)
    want = owner_gathers(p, kernel, op)
    assert want == (not soa if gather is None else gather)
    o = oracle_of(p, kernel)
    O.loop_owner_replay(o, op, 2)
    stats = p.gpu_loop(f, capi.STRATEGY_HIERARCHICAL, 2, block_size=bs, flags=capi.LOOP_OWNER_COMPUTE)
    assert stats["lds_bytes"] == owner_lds(p, op, want), stats
    assert_bitwise(p.point_data[0], o.target, f"{kind} {parts}")


# ---- atomics -------------------------------------------------------------------
@pytest.mark.gpu
@pytest.mark.parametrize("soa", [False, True])
@pytest.mark.parametrize("order", [None, "gps"])
@pytest.mark.parametrize("kind,n", [("hex", 12), ("hex", 24), ("hex", 30), ("getacc", 50),
                                    ("getacc", 112), ("mine8", 14), ("mine8", 27), ("mine8", 43)])
def test_atomics_by_themselves_and_in_the_table(gpu, kind, n, order, soa):
    """The atomics loop on either side of the sizes where small meshes of cells
    with four or eight points leave the table out, ordered and shuffled."""
    points = n + 1
    if kind == "getacc":
        p, kernel, f = getacc_problem(points, points, soa=soa), O.GETACC, \
            capi.functor(capi.KERNEL_GETACC)
    else:
        cells = meshgen.hex_grid(points, points, points)
        cells = cells[meshgen.permutation(cells.shape[0], 3)]
        td = 3 if kind == "hex" else 4
        pd = meshgen.uniform(td * points ** 3, 1).reshape(-1, td)
        data = meshgen.normal(cells.shape[0] * (24 if kind == "hex" else 4), 2)
        p = Problem([cells], [points ** 3], [pd.T.copy() if soa else pd],
                    [data.reshape(-1, cells.shape[0])], 128, soa)
        kernel = O.HEX_SCATTER if kind == "hex" else O.MINE8
        f = capi.functor(capi.KERNEL_HEX_SCATTER) if kind == "hex" else \
            capi.functor(capi.KERNEL_MINE, 8, 4, 4)
    if order:
        p.reorder(order)
    o = oracle_of(p, kernel)
    scale = o.loop_serial(1, with_scale=True)
    p.gpu_loop(f, capi.STRATEGY_ATOMIC, 1, block_size=96)
    assert_close_scaled(p.point_data[0], o.target, scale, what=f"{kind} {n}")


# ---- the gathering kernels of each functor --------------------------------------
NT = capi.LOOP_NONTEMPORAL
STAGE = capi.LOOP_STAGE_INPUTS


def element_problem(kind, n, soa):
    if kind == "lulesh":
        return lulesh_problem(n + 1, n, n + 2, soa=soa), O.LULESH, capi.functor(capi.KERNEL_LULESH)
    if kind == "getacc":
        return getacc_problem(5 * n, 4 * n, soa=soa), O.GETACC, capi.functor(capi.KERNEL_GETACC)
    return hex_problem(n, soa=soa), O.HEX_SCATTER, capi.functor(capi.KERNEL_HEX_SCATTER)


@pytest.mark.gpu
@pytest.mark.parametrize("soa", [False, True])
@pytest.mark.parametrize("kind,n,method,block_size,gather", [
    ("hex", 13, "bisect", 256, True), ("hex", 13, "bisect", 128, False),
    ("hex", 9, None, 128, False), ("lulesh", 13, "bisect", 512, True),
    ("lulesh", 13, "bisect", 256, True), ("lulesh", 13, None, 256, False),
    ("getacc", 12, "bisect", 128, True), ("getacc", 12, "bisect", 512, True),
    ("getacc", 14, None, 256, False)])
def test_element_loops_gather_on_compact_parts(gpu, kind, n, method, block_size, gather, soa):
    """hex, lulesh and getacc on parts that gather and on blocks with too many
    points that do not: per colour, two-phase and with nontemporal cell data,
    bits of the oracle's replay; lulesh's volumes come from either kernel."""
    p, kernel, f = element_problem(kind, n, soa)
    p.block_size = block_size
    if method:
        p.partition(method=method)
        p.reorder_to_partition()
        p.renumber_points()
    flags = (0, TP, TP | NT) if kind != "getacc" else (0, TP)
    volumes = None
    if kind == "lulesh":
        o = oracle_of(p, kernel)
        o.loop_serial(1)
        volumes = np.array(o.cell_data[1])
    for iters in (1, 2):
        q = copy.deepcopy(p)
        for fl in flags:
            check(q, kernel, f, block_size, iters, gather, (fl,))
            if volumes is not None:
                assert_bitwise(q.cell_data[1], volumes, f"volumes, flags {fl}")
                q.cell_data[1][:] = np.nan
            q.point_data = copy.deepcopy(p.point_data)


# ---- lists of exactly 4, 8 and 9 increments in a block ---------------------------
def hub_blocks(degree, blocks=5):
    """Edges in blocks of 64, every block a bipartite graph of its own first points
    and of second points it shares with its neighbour, whose first points have
    `degree` edges; (edges, points)."""
    per = 64 // degree                    # first points a block
    edges = []
    for b in range(blocks):
        first = np.repeat(np.arange(per), degree)
        second = (first + np.tile(np.arange(degree), per)) % max(per, degree)
        e = np.stack([32 * b + first, 1000 + 40 * (b // 2) + second], 1)
        rest = 64 - e.shape[0]            # (degree 9: one more edge of two points more)
        extra = np.stack([32 * b + 20 + np.arange(rest), 1000 + 40 * (b // 2) + 30 + np.arange(rest)], 1)
        block = np.concatenate([e, extra])
        edges.append(block[np.random.default_rng(b).permutation(64)])
    edges = np.concatenate(edges)
    ids, at = np.unique(edges, return_inverse=True)
    return at.reshape(edges.shape).astype(np.uint32), ids.size


@pytest.mark.gpu
@pytest.mark.parametrize("soa", [False, True])
@pytest.mark.parametrize("degree", [4, 8, 9])
def test_hierarchical_lists_of_4_8_and_9(gpu, degree, soa):
    maps, n = hub_blocks(degree)
    pd = meshgen.uniform(4 * n, 1).reshape(n, 4)
    p = Problem([maps], [n], [pd.T.copy() if soa else pd],
                [meshgen.uniform(4 * maps.shape[0], 2).reshape(4, -1)], 64, soa)
    h = check(p, O.MINE2, capi.functor(capi.KERNEL_MINE, 2, 4, 4), 64, 2, degree <= 8)
    assert h["longest"] == degree and h["threads"] == 64


def staged_check(p, gather, block_size, iters=2):
    """Staged res_calc per colour and two-phase against the replay, on the kernel
    expected."""
    h = host_plan(p, block_size)
    assert gather == (h["blocks"] < 1024 and h["longest"] <= 8 and h["most"] <= 2 * h["threads"])
    o = oracle_of(p, O.RES_CALC)
    o.loop_hier_replay(O.OraclePlan(p.maps, p.num_points[0], block_size, p.partition_vector), iters)
    start = [d.copy() for d in p.point_data]
    for fl in (STAGE, STAGE | TP):
        p.point_data = [d.copy() for d in start]
        stats = p.gpu_loop(capi.functor(capi.KERNEL_RES_CALC), capi.STRATEGY_HIERARCHICAL, iters,
                           block_size=block_size, flags=fl)
        lds = 8 * max(5 * h["most"], 4 * (h["threads"] + 1)) if gather else 72 * h["most"]
        assert stats["lds_bytes"] == lds, (stats, h)
        assert_bitwise(p.point_data[0], o.target, f"flags {fl} {h}")
    return h


@pytest.mark.gpu
@pytest.mark.parametrize("soa", [False, True])
@pytest.mark.parametrize("degree", [4, 8, 9])
def test_staged_res_calc_lists_of_4_8_and_9(gpu, degree, soa):
    maps, n = hub_blocks(degree)
    rng = np.random.default_rng(degree)
    q = np.array([1.0, 0.4, 0.0, 2.5]) * (1 + 1e-2 * rng.normal(size=(n, 4)))
    res, x, adt = rng.normal(size=(n, 4)), rng.normal(size=(50, 2)), rng.uniform(0.5, 1.5, n)
    nodes = rng.integers(0, 50, maps.shape).astype(np.uint32)
    if soa:
        res, x, q = res.T.copy(), x.T.copy(), q.T.copy()
    p = Problem([maps, nodes, maps, maps], [n, 50, n, n], [res, x, q, adt], (), 64, soa)
    assert staged_check(p, degree <= 8, 64)["longest"] == degree


@pytest.mark.gpu
@pytest.mark.parametrize("soa", [False, True])
@pytest.mark.parametrize("nx,ny,gather", [(236, 139, True), (240, 140, False)])
def test_staged_res_calc_on_either_side_of_1024_blocks(gpu, nx, ny, gather, soa):
    p = airfoil_problem(nx, ny, soa=soa, res0_seed=4)
    p.reorder("gps")
    h = staged_check(p, gather, 64, 1)
    assert 1000 <= h["blocks"] < 1060

"""fot_loop_run's first and last steps against steps with explicit copies,
over the kernels that have a form of their own for them."""
import numpy as np
import pytest

from cuda_fot_amd import DeviceArray, Loop, capi, lulesh_problem
from helpers import airfoil_problem, assert_bitwise, mine_problem

pytestmark = pytest.mark.gpu

OWN = capi.LOOP_OWNER_COMPUTE
GATHER = OWN | capi.LOOP_OWNER_GATHER


def run_and_steps(p, f, flags, iters, jacobi, partition=None, block_size=128):
    """(iterate, output) after run(iters), then the same by steps and copies."""
    got = []
    for whole in (True, False):
        dev = [DeviceArray.from_host(d) for d in p.point_data]
        out = DeviceArray.from_host(np.full_like(p.point_data[0], np.nan))
        cells = [DeviceArray.from_host(c) for c in p.cell_data]
        loop = Loop(f, p.maps, p.num_points, dev, out, cells, soa=p.soa, block_size=block_size,
                    partition=partition, flags=flags)
        if whole:
            loop.run(iters)
        else:
            capi.call("fot_copy", out.ptr, dev[0].ptr, out.nbytes, None)
            for i in range(iters):
                loop.step()
                if jacobi or i + 1 == iters:
                    capi.call("fot_copy", dev[0].ptr, out.ptr, out.nbytes, None)
        got += [dev[0].download(), out.download()]
        loop.close()
    return got


@pytest.mark.parametrize("soa", [False, True])
@pytest.mark.parametrize("form", [0, capi.LOOP_PERSISTENT, capi.LOOP_POINT_TERMS,
                                  capi.LOOP_LISTS_IN_HBM, capi.LOOP_NONTEMPORAL])
@pytest.mark.parametrize("two", [0, capi.LOOP_TWO_PER_THREAD])
def test_owner_res_calc_run_forms(gpu, form, two, soa):
    p = airfoil_problem(nx=40, ny=26, soa=soa, res0_seed=5)
    for iters in (1, 2, 3):
        got = run_and_steps(p, capi.functor(capi.KERNEL_RES_CALC), GATHER | two | form, iters, False)
        for g in got[:3]:
            assert_bitwise(g, got[3], f"form {form} two {two} iters {iters}")


@pytest.mark.parametrize("soa", [False, True])
@pytest.mark.parametrize("flags", [OWN, capi.LOOP_TWO_PHASE,
                                   capi.LOOP_TWO_PHASE | capi.LOOP_STAGE_INPUTS])
@pytest.mark.parametrize("order", [None, "gps"])  # AOS two-phase: gathered sums, colour loop
def test_mine_run_forms(gpu, order, flags, soa):
    p = mine_problem(N=90, M=57, soa=soa, shuffle=False)
    if order:
        p.reorder(order)
    else:
        p.partition(method="bisect")
        p.reorder_to_partition()
        p.renumber_points()
    for iters in (1, 3):
        got = run_and_steps(p, capi.functor(capi.KERNEL_MINE, 2, 4, 4), flags, iters, True,
                            None if order else p.partition_vector)
        for g in got[:3]:
            assert_bitwise(g, got[3], f"flags {flags} iters {iters}")


class Place:
    """Part of another buffer, as a loop takes an array."""

    def __init__(self, buffer, first, shape):
        self.buffer, self.ptr, self.shape = buffer, buffer.ptr + 8 * first, shape


@pytest.mark.parametrize("iters", [1, 2])
def test_run_whose_output_is_another_input(gpu, iters):
    """The output is the buffer of the node coordinates, which the loop reads:
    the copy into it comes before the first step."""
    p = lulesh_problem(5, 4, 6, block_size=32)
    f = capi.functor(capi.KERNEL_LULESH)
    got = []
    for whole in (True, False):
        force, xyz = (DeviceArray.from_host(d) for d in p.point_data)
        cells = [DeviceArray.from_host(c) for c in p.cell_data]
        loop = Loop(f, p.maps, p.num_points, [force, xyz], xyz, cells, block_size=32,
                    flags=capi.LOOP_TWO_PHASE)
        if whole:
            loop.run(iters)
        else:
            capi.call("fot_copy", xyz.ptr, force.ptr, xyz.nbytes, None)
            for _ in range(iters):
                loop.step()
            capi.call("fot_copy", force.ptr, xyz.ptr, xyz.nbytes, None)
        got.append((force.download(), xyz.download()))
        loop.close()
    for a, b in zip(*got):
        assert_bitwise(a, b, f"iters {iters}")


@pytest.mark.parametrize("iters", [1, 2])
@pytest.mark.parametrize("inside", ["output", "iterate", "coordinates"])
def test_run_whose_cell_output_lies_in_point_data(gpu, inside, iters):
    """The element volumes are written inside another array: after every step
    has read and written it."""
    p = lulesh_problem(5, 4, 6, block_size=32)
    f, nc = capi.functor(capi.KERNEL_LULESH), p.num_cells
    got = []
    for overlap in (True, False):
        force, xyz = (DeviceArray.from_host(d) for d in p.point_data)
        out = DeviceArray.from_host(np.zeros_like(p.point_data[0]))
        sigma = DeviceArray.from_host(p.cell_data[0])
        into = dict(output=out, iterate=force, coordinates=xyz)[inside]
        volume = Place(into, 7, (1, nc)) if overlap else DeviceArray.from_host(p.cell_data[1])
        loop = Loop(f, p.maps, p.num_points, [force, xyz], out, [sigma, volume], block_size=32,
                    flags=capi.LOOP_TWO_PHASE)
        loop.run(iters)
        arrays = dict(iterate=force.download(), output=out.download(), coordinates=xyz.download())
        if not overlap:
            arrays[inside].reshape(-1)[7:7 + nc] = volume.download().reshape(-1)
        got.append(arrays)
        loop.close()
    for k in got[0]:
        assert_bitwise(got[0][k], got[1][k], f"{k}, volumes in {inside}")


@pytest.mark.parametrize("aligned", [True, False])
def test_owner_res_calc_run_on_an_iterate_of_any_alignment(gpu, aligned):
    """An iterate that starts on an odd multiple of 8 bytes: the copies take it,
    the step's 16-byte loads and stores do not touch it."""
    p = airfoil_problem(nx=20, ny=13, res0_seed=5)
    n = p.point_data[0].size
    dev = [DeviceArray.from_host(d) for d in p.point_data]
    room = DeviceArray.from_host(np.concatenate([[7.0], p.point_data[0].reshape(-1), [9.0]]))
    if not aligned:
        dev[0] = Place(room, 1, p.point_data[0].shape)
        assert dev[0].ptr % 16 == 8
    out = DeviceArray.from_host(np.full_like(p.point_data[0], np.nan))
    loop = Loop(capi.functor(capi.KERNEL_RES_CALC), p.maps, p.num_points, dev, out, (),
                block_size=128, flags=GATHER | capi.LOOP_TWO_PER_THREAD)
    loop.run(2)
    got = dev[0].download() if aligned else room.download()[1:n + 1].reshape(-1, 4)
    ref = run_and_steps(p, capi.functor(capi.KERNEL_RES_CALC), GATHER | capi.LOOP_TWO_PER_THREAD,
                        2, False)[3]
    assert_bitwise(got, ref, "iterate")
    assert_bitwise(out.download(), ref, "output")
    if not aligned:
        assert room.download()[0] == 7.0 and room.download()[n + 1] == 9.0
    loop.close()


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("stage", [0, capi.LOOP_STAGE_INPUTS])
def test_dependency_ordered_blocks_see_their_predecessors(gpu, stage, graph):
    """Many small blocks that share cache lines over all XCDs, run after run: a
    block adds to what its predecessors wrote, never to an older value."""
    p = airfoil_problem(110, 100, seed=3, block_size=32)
    p.reorder("gps")
    f = capi.functor(capi.KERNEL_RES_CALC)
    dev = [DeviceArray.from_host(d) for d in p.point_data]
    out = DeviceArray.from_host(np.zeros_like(p.point_data[0]))
    got = []
    for flags in (stage, stage | capi.LOOP_DEPENDENCY_ORDER):
        loop = Loop(f, p.maps, p.num_points, dev, out, (), block_size=32, flags=flags,
                    use_graph=graph)
        for _ in range(1 if flags == stage else 400):
            dev[0].upload(p.point_data[0])
            loop.run(2)
            got.append(dev[0].download())
        loop.close()
    for i, g in enumerate(got[1:]):
        assert_bitwise(g, got[0], f"run {i}")

"""fot_loop_run's first and last steps against steps with explicit copies,
over the kernels that have a form of their own for them."""
import numpy as np
import pytest

from cuda_fot_amd import DeviceArray, Loop, capi
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
@pytest.mark.parametrize("flags", [OWN, capi.LOOP_TWO_PHASE])
def test_mine_run_forms(gpu, flags, soa):
    p = mine_problem(N=30, M=17, soa=soa)
    for iters in (1, 3):
        got = run_and_steps(p, capi.functor(capi.KERNEL_MINE, 2, 4, 4), flags, iters, True)
        for g in got[:3]:
            assert_bitwise(g, got[3], f"flags {flags} iters {iters}")

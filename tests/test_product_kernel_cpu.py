"""Which kernel a plain product runs (eh_plan_kernel): the planner's other modes
and an installed network keep their configuration."""
import ctypes as C

import numpy as np
import pytest

import eigen_amd as E
from oracle import mlp as M


@pytest.fixture
def default_planner():
    prev = E.lib().eh_get_tune_mode()
    E.set_tune_mode(E.TUNE_MLP)
    yield
    E.set_tune_mode(prev)


def test_kernels_of_the_default_planner(default_planner):
    for dt in (E.F32, E.F64):
        assert E.plan_kernel(dt, 0, 0, 96, 80, 112) == E.KERNEL_SMALL
        assert E.plan_kernel(dt, 0, 0, 1, 80, 112) == E.KERNEL_VECTOR
        assert E.plan_kernel(dt, 1, 0, 80, 1, 112) == E.KERNEL_VECTOR
        assert E.plan_kernel(dt, 0, 0, 4096, 4096, 4096) == E.KERNEL_CONFIG
    assert E.plan_kernel(E.F64, 1, 0, 1000, 777, 1203) == E.KERNEL_BALANCED


def test_other_planners_keep_their_configuration(default_planner):
    E.set_tune_mode(E.TUNE_HEURISTIC)
    assert E.plan_kernel(E.F64, 0, 0, 96, 80, 112) == E.KERNEL_CONFIG
    assert E.plan_kernel(E.F64, 1, 0, 1000, 777, 1203) == E.KERNEL_CONFIG
    E.set_tune_mode(E.TUNE_MLP)
    params = np.zeros(M.N_PARAMS, np.float32)
    E.check(E.lib().eh_planner_set_mlp_params(params.ctypes.data_as(C.c_void_p)))
    try:
        assert E.plan_kernel(E.F64, 1, 0, 1000, 777, 1203) == E.KERNEL_CONFIG
    finally:
        E.check(E.lib().eh_planner_set_mlp_params(None))
    assert E.plan_kernel(E.F64, 1, 0, 1000, 777, 1203) == E.KERNEL_BALANCED


def test_argument_checks():
    for bad in ((7, 0, 0, 2, 2, 2), (E.F64, 5, 0, 2, 2, 2), (E.F64, 0, 0, 0, 2, 2), (E.F64, 0, 0, 2, 2, 0)):
        with pytest.raises(E.EigenAmdError):
            E.plan_kernel(*bad)


@pytest.mark.parametrize("dt,ta,tb,m,n,k,want", [
    # few tiles whose many parts one workgroup would add up one after another
    (E.F64, 1, 0, 64, 64, 2048, 0), (E.F64, 1, 0, 366, 22, 5844, 0), (E.F64, 1, 0, 11, 7, 34727, 0),
    (E.F32, 1, 1, 5, 270, 2107, 0), (E.F32, 0, 0, 2, 443, 1663, 0), (E.F32, 1, 0, 688, 55, 1759, 0),
    # runs of about a tile: every tile cut, nothing balanced
    (E.F64, 0, 1, 2683, 1057, 2702, 0), (E.F64, 1, 1, 2959, 1551, 2262, 0), (E.F32, 1, 0, 903, 1358, 409, 0),
    (E.F32, 1, 0, 523, 1871, 385, 0), (E.F64, 0, 0, 2049, 701, 2999, 0),
    # what the balanced kernel is for
    (E.F64, 1, 0, 1000, 777, 1203, 1), (E.F32, 0, 0, 779, 796, 1129, 1), (E.F64, 0, 0, 130, 130, 20000, 1)])
def test_balanced_only_where_it_was_measured_faster(default_planner, dt, ta, tb, m, n, k, want):
    assert (E.plan_kernel(dt, ta, tb, m, n, k) == E.KERNEL_BALANCED) == bool(want)

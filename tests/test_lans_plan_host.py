"""What LansPlan.step refuses before it reaches the native call, without a GPU."""
import ctypes as C
import importlib

import pytest

pkg = importlib.import_module("lancet-accelerating-moe-training-via-whole-graph-computation-communication-overlapping_amd")


class _Other(C.Structure):
    _fields_ = [("lr", C.c_float)]


def _plan():
    plan = object.__new__(pkg.ops.LansPlan)
    plan.numels, plan._sizes, plan._h, plan._lib = [], 0, C.c_void_p(1), None
    return plan


@pytest.mark.parametrize("hyper", [None, _Other(1e-3), C.c_float(1.0), 0, "x", C.pointer(_Other())])
def test_another_structure_is_refused(hyper):
    plan = _plan()
    try:
        with pytest.raises(TypeError, match="LansHyper"):
            plan.step([], [], [], [], 1, hyper)
    finally:
        plan._h = None


def test_a_closed_plan_is_refused():
    plan = _plan()
    plan._h = None
    with pytest.raises(pkg.capi.LancetError) as info:
        plan.step([], [], [], [], 1, pkg.capi.LansHyper())
    assert info.value.status == pkg.capi.ERR_PLAN

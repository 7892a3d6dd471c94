"""Scratch of block-contraction plans: a cached plan is shared by every stream and thread that
contracts the same structure, so two executions that are in flight must not share scratch."""
import ctypes

from cytnx_amd.unitensor import CPU, _Plan


def _plan(nbytes):
    p = _Plan.__new__(_Plan)  # metadata only: plans themselves are made on a device
    p.handle, p.device, p.ws_bytes, p._ws = 0, CPU, nbytes, None
    return p


def _address(arg):
    return ctypes.c_void_p.from_param(arg), ctypes.cast(
        getattr(arg, "_as_parameter_", arg) or 0, ctypes.c_void_p).value


def test_executions_in_flight_have_their_own_scratch():
    p = _plan(4096)
    first, second = p.workspace(), p.workspace()
    (_, a), (_, b) = _address(first), _address(second)
    assert a and b
    assert abs(a - b) >= 4096


def test_plans_without_scratch_pass_null():
    assert not _plan(0).workspace()

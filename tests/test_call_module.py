"""The module that takes Plan.gemm and Plan.lstm_step to the library without ctypes (csrc/tw_call.cpp): plain arguments arrive
as ctypes would hand them over, any other makes it stand aside."""
import ctypes
import os
import subprocess
import sys
import sysconfig

import numpy as np
import pytest

GEMM_ARGS = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_void_p, ctypes.c_int, ctypes.c_int64,
             ctypes.c_int, ctypes.c_float, ctypes.c_float, ctypes.c_int, ctypes.c_void_p]


@pytest.fixture
def calls(tw):
    """The module bound to Python functions that write down what arrives, and back to the library afterwards."""
    from tilesparsity_amd import _twcall
    tw.lib()
    seen = []

    def gemm(kind, n_more):
        def f(plan, A, a_layout, lda, C, c_layout, ldc, M, alpha, beta, pruned, ep, *rest):
            seen.append((kind, plan, A, a_layout, lda, C, c_layout, ldc, M, alpha, beta, pruned,
                         ep[0].bias, ep[0].activation) + rest)
            return -3
        types = GEMM_ARGS[:11] + [ctypes.POINTER(tw.Epilogue)] + [ctypes.c_void_p, ctypes.c_int64][:n_more] + [ctypes.c_void_p]
        return ctypes.CFUNCTYPE(ctypes.c_int, *types)(f)

    def step(*args):
        seen.append(("step",) + args)
        return 0
    vp, i64, i, f = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int, ctypes.c_float
    fns = [gemm("ex", 0), gemm("static", 0), gemm("staged", 2),
           ctypes.CFUNCTYPE(i, vp, vp, i64, i, vp, f, vp, i64, vp, i64, vp, i64, vp, i64, vp)(step)]
    L = tw.lib()
    real = [ctypes.cast(getattr(L, n), vp).value for n in ("tw_gemm_ex", "tw_gemm_static", "tw_gemm_staged", "tw_lstm_step")]
    _twcall.bind(*(ctypes.cast(fn, vp).value for fn in fns))
    yield _twcall, seen
    _twcall.bind(*real)


def test_arguments_arrive(calls):
    mod, seen = calls
    big = 0x7F0123456780
    plain = [big, big + 16, 0, 1 << 40, None, 1, -8, 7, 0.5, 2, 1, big + 64, None, 2, False, None, 0]
    assert mod.gemm(*plain) == -3
    assert seen.pop() == ("ex", big, big + 16, 0, 1 << 40, None, 1, -8, 7, 0.5, 2.0, 1, None, 2, big + 64)
    assert mod.gemm(*(plain[:14] + [True] + plain[15:])) == -3 and seen.pop()[0] == "static"
    assert mod.gemm(*(plain[:12] + [big + 128, 1, False, big + 256, 1 << 33])) == -3
    got = seen.pop()
    assert got[0] == "staged" and got[12:] == (big + 128, 1, big + 256, 1 << 33, big + 64)
    # the low bits, as ctypes takes them
    assert mod.gemm(*(plain[:7] + [(1 << 32) + 5] + plain[8:])) == -3 and seen.pop()[8] == 5
    args = [big, big + 2, 64, 5, None, 1, big + 4, 72, big + 6, 80, big + 8, 88, None, 96, None]
    assert mod.lstm_step(*args) == 0
    assert seen.pop() == tuple(["step"] + args[:5] + [1.0] + args[6:])


@pytest.mark.parametrize("at,value", [(7, 5.0), (3, np.int64(8)), (8, "1"), (1, ctypes.c_void_p(16)), (13, np.int32(1)),
                                      (14, 1), (8, 10 ** 400), (7, True)])
def test_other_arguments_are_left_to_ctypes(calls, at, value):
    mod, seen = calls
    args = [16, 16, 0, 8, 16, 0, 8, 1, 1.0, 0.0, 0, 0, None, 0, False, None, 0]
    args[at] = value
    assert mod.gemm(*args) is None and not seen
    assert mod.gemm(*args[:5]) is None and mod.lstm_step(*args) is None and not seen


def test_a_destroyed_plan_is_refused(tw):
    plan = tw.Plan(0, 64, 64, 0)
    with pytest.raises(tw.TwError) as e:
        plan.gemm(16, 16, 8)
    assert e.value.status == tw.ERR_NULL
    with pytest.raises(tw.TwError):
        plan.lstm_step(16, 8, 16, 16, 16)
    with pytest.raises(ctypes.ArgumentError):
        plan.gemm(16, 16, 8.5, lda=8, ldc=8)


def test_the_library_without_the_module(tw):
    """A tree without the module, or with one that another interpreter built: all calls go through ctypes, as a warning says."""
    code = r"""
import sys, warnings
sys.modules["tilesparsity_amd._twcall"] = None
from tilesparsity_amd import twgemm as tw
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    assert tw.lib() is tw.lib()
assert len(seen) == 1 and "ctypes" in str(seen[0].message), seen
plan = tw.Plan(0, 64, 64, 0)
for call in (lambda: plan.gemm(16, 16, 8), lambda: plan.gemm(16, 16, 8, workspace_ptr=16, workspace_bytes=64),
             lambda: plan.gemm(16, 16, 8, static=True), lambda: plan.lstm_step(16, 8, 16, 16, 16)):
    try:
        call()
    except tw.TwError as e:
        assert e.status == tw.ERR_NULL
    else:
        raise AssertionError
"""
    subprocess.run([sys.executable, "-c", code], check=True, cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))


def test_the_module_is_this_interpreters(tw):
    """Its name says which interpreter it was built for: another one does not load it."""
    from tilesparsity_amd import _twcall, build
    assert _twcall.__file__ == build.CALL_PATH and _twcall.__file__.endswith(sysconfig.get_config_var("EXT_SUFFIX"))
    assert not os.path.exists(os.path.join(build.PKG_DIR, "_twcall.so"))

"""Launch binding without the inspect module's signatures binds as it does, and
annotations follow the names they use."""

from __future__ import annotations

import copy
import inspect
import pickle

import numpy as np
import pytest

from hc import LaunchError
from hc._launch import _bind_arguments, buffer_dtype_name, resolved_annotations
from hc.core import Buffer
from hc.symbols import sym


def _plain(group, a, b, c):
    pass


def _defaults(group, a, b=2):
    pass


def _variadic(group, a, *rest, **more):
    pass


def _keyword_only(group, a, *, b):
    pass


def _wrapped(group, *args):
    pass


_wrapped.__wrapped__ = _plain


@pytest.mark.parametrize("fn,args,kwargs", [
    (_plain, (1, 2, 3), {}), (_plain, (1, 2), {"c": 3}), (_defaults, (1,), {}), (_defaults, (1, 5), {}),
    (_variadic, (1, 2, 3), {"z": 4}), (_variadic, (1,), {}), (_keyword_only, (1,), {"b": 2}), (_wrapped, (1, 2, 3), {}),
])
def test_binding_equals_inspect(fn, args, kwargs):
    want = inspect.Signature(list(inspect.signature(fn).parameters.values())[1:]).bind(*args, **kwargs)
    got = _bind_arguments(fn, args, kwargs)
    assert got.arguments == want.arguments and list(got.arguments) == list(want.arguments)
    assert got.args == want.args and got.kwargs == want.kwargs and got.signature == want.signature


@pytest.mark.parametrize("fn,args", [(_plain, (1, [2], 3)), (_defaults, (1,))])
def test_bound_arguments_copy_and_pickle(fn, args):
    """A lowering may keep a copy of the arguments it was given."""
    bound = _bind_arguments(fn, args, {})
    shallow = copy.copy(bound)
    assert shallow == bound and shallow.arguments["a"] is bound.arguments["a"]
    for other in (copy.deepcopy(bound), pickle.loads(pickle.dumps(bound))):
        assert other == bound and other.args == args and other.signature == bound.signature


@pytest.mark.parametrize("args,kwargs", [((1, 2), {}), ((1, 2, 3, 4), {}), ((1, 2, 3), {"c": 4}), ((1, 2, 3), {"d": 4})])
def test_binding_refuses_what_inspect_refuses(args, kwargs):
    with pytest.raises(LaunchError, match="cannot bind launch arguments"):
        _bind_arguments(_plain, args, kwargs)
    with pytest.raises(LaunchError, match="CurrentGroup"):
        _bind_arguments(lambda: None, (), {})


DT = np.float16


def test_string_annotations_follow_globals_closures_and_symbols():
    global DT
    width = 16

    def kernel(group, a: Buffer[M, width, DT], b: Buffer[Rows, 8]):  # noqa: F821
        return width

    first = resolved_annotations(kernel)
    assert first["a"].dimensions == (sym.M, 16) and first["a"].dtype == "float16"
    assert first["b"].dimensions == (sym.Rows, 8)
    width = 32
    DT = np.float32
    try:
        again = resolved_annotations(kernel)
    finally:
        DT = np.float16
    assert again["a"].dimensions == (sym.M, 32) and again["a"].dtype == "float32"
    kernel.__annotations__["b"] = "  Buffer[Rows, 8]"
    assert resolved_annotations(kernel)["b"].dimensions == (sym.Rows, 8)
    kernel.__annotations__["b"] = "Buffer[lower, 8]"
    with pytest.raises(LaunchError, match="failed to resolve annotations"):
        resolved_annotations(kernel)


def test_dtype_names():
    torch = pytest.importorskip("torch")
    for _ in range(2):
        assert buffer_dtype_name(torch.empty(1, dtype=torch.bfloat16)) == "bfloat16"
        assert buffer_dtype_name(np.empty(1, np.float16)) == "float16"
        assert buffer_dtype_name([1.0]) is None
    assert Buffer[sym.M, np.longdouble].dtype == np.dtype(np.longdouble).name
    assert Buffer[sym.M, 4].dtype is None

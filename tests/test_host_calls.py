"""The native callables behind the Python face (csrc/python_calls.cc) against ctypes: same results and codes, and what they do
not take is left to ctypes.  Dry worlds: nothing here touches a GPU."""
import copy
import ctypes
import enum
import functools
import inspect
import os
import pickle
import subprocess
import sys
import sysconfig
import threading
import types
import weakref

import pytest

from hccl_amd import _lib, api
from hccl_amd import types as T


class Kind(enum.IntEnum):
    FP32 = T.FP32


@pytest.fixture(scope="module")
def world():
    w = api.World(2, dry=True)
    yield w
    w.close()


@pytest.mark.parametrize("args", [(0, 2, 10, 4, 0, "comm", 1), (1, 2, 10, 99, 0, "comm", 1), (1, 2, 10, 4, 9, "comm", 1),
                                  (1, 2, 1 << 63, 4, 0, "comm", 1), (1, 2, -1, 4, 0, "comm", 1), (1, 2, 10, 4, 0, 0, 1),
                                  (1, 2, 10, 4, 0, "comm", 0), (None, 2, 10, 4, 0, "comm", 1), (1, 2, (1 << 64) + 10, 4 + (1 << 32), 9, "comm", 1)])
def test_codes_are_those_of_ctypes(world, args):
    args = [world.comms[0] if a == "comm" else a for a in args]
    native = api._all_reduce(*args)
    assert native == api.lib().HcclAllReduce(*args) and native != 0


@pytest.mark.parametrize("args", [(1.5, 2, 10, 4, 0, 7, 1), ([1, 2], 2, 10, 4, 0, 7, 1), (ctypes.c_void_p(5), 2, 10, 4, 0, 7, 1),
                                  (1, 2, None, 4, 0, 7, 1), (1, 2, 10, None, 0, 7, 1), (1, 2, (ctypes.c_uint64 * 2)(), 4, 0, 7, 1),
                                  (b"x", 2, 10, 4, 0, 7, 1)])
def test_other_types_are_left_to_ctypes(world, args):
    assert api._all_reduce(*args) is NotImplemented


def test_what_ctypes_refuses_is_refused(world):
    for bad in ([1, 2], 1.5):
        with pytest.raises(ctypes.ArgumentError):
            world.all_reduce(0, bad, 2 << 20, 10, T.FP32, T.SUM, 1)
    with pytest.raises(ctypes.ArgumentError):
        world.all_reduce(0, 1 << 20, 2 << 20, None, T.FP32, T.SUM, 1)
    with pytest.raises(TypeError):
        api._all_reduce(1, 2, 3)


def test_enumerations_and_addresses_in_ctypes_objects(world):
    for r in range(2):
        assert world.all_reduce(r, ctypes.c_void_p((r + 1) << 20), (r + 10) << 20, 100, Kind.FP32, T.SUM, 1) == 0
    assert world.last_info().algName


def test_tables_as_lists_and_as_converted_arrays(world):
    for table in (list, api.u64_table):
        for r in range(2):
            assert world.all_to_all_v(r, (r + 1) << 20, table([3, 4]), table([0, 3]), (r + 10) << 20, table([3 + r, 3 + r]),
                                      table([0, 3 + r]), T.FP32, 1) == 0
            assert world.all_gather_v(r, (r + 1) << 20, 5 + r, (r + 10) << 20, table([5, 6]), table([0, 5]), T.FP32, 1) == 0


def test_the_callable_from_several_threads(world):
    """The interpreter lock is given up during the call: ranks may call from threads of their own."""
    codes = []
    def rank(r):
        for _ in range(50):
            codes.append(world.all_reduce(r, (r + 1) << 20, (r + 10) << 20, 100, T.FP32, T.SUM, 1))
    threads = [threading.Thread(target=rank, args=(r,)) for r in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert codes == [0] * 100


def test_pointer_lists():
    call = _lib.native_call("hcclx_moe_route")
    assert call([1] * 65, 65, 8, 8, 1, 1, 1, 1, [1] * 65, 1, 0) is NotImplemented
    assert call(1, 1, 8, 8, 1, 1, 1, 1, [1], 1, 0) is NotImplemented
    assert call([1.5], 1, 8, 8, 1, 1, 1, 1, [1], 1, 0) is NotImplemented


ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_without_the_module_the_calls_go_through_ctypes():
    """The library alone is enough: the module may not have been built (no Python headers) or be another interpreter's."""
    code = """
from hccl_amd import _lib, api, types as T
_lib.CALLS_PATH += ".missing"
w = api.World(2, dry=True)
assert api._all_reduce(1, 2, 10, T.FP32, T.SUM, w.comms[0], 1) is NotImplemented
for r in range(2):
    assert w.all_reduce(r, (r + 1) << 20, (r + 10) << 20, 100, T.FP32, T.SUM, 1) == 0
    assert w.all_to_all(r, (r + 1) << 20, 5, (r + 10) << 20, T.FP32, 1) == 0
    assert w.all_to_all_v(r, (r + 1) << 20, [3, 4], [0, 3], (r + 10) << 20, [3 + r, 3 + r], [0, 3 + r], T.FP32, 1) == 0
assert w.last_info().algName
w.close()
"""
    run = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stderr[-2000:]


def test_the_module_is_named_after_the_interpreter_it_was_built_for():
    name = "_hccl_calls" + sysconfig.get_config_var("EXT_SUFFIX")
    assert os.path.basename(_lib.CALLS_PATH) == name and os.path.exists(_lib.CALLS_PATH)


@pytest.mark.parametrize("headers", [True, False])
def test_the_build_needs_no_python_headers(tmp_path, headers):
    """An interpreter that names a header directory: the module is built for its ABI where Python.h is in there."""
    if headers:
        (tmp_path / "Python.h").write_text("")
    python = tmp_path / "python"
    python.write_text(f"""#!/bin/sh
case "$2" in *EXT_SUFFIX*) echo .cpython-399-test.so;; *) echo {tmp_path};; esac
""")
    python.chmod(0o755)
    csrc = os.path.join(ROOT, "hccl_amd", "csrc")
    run = subprocess.run(["make", "-n", "-C", csrc, f"PYTHON={python}", f"LIBDIR={tmp_path}/lib", "all"], capture_output=True, text=True)
    assert run.returncode == 0, run.stderr[-2000:]
    assert "libhccl_amd.so" in run.stdout
    assert ("_hccl_calls.cpython-399-test.so" in run.stdout) == headers and ("python_calls.cc" in run.stdout) == headers


@pytest.mark.parametrize("how", ["plain", "keywords", "unbound", "kind", "boolean rank", "subclass"])
def test_the_native_methods_and_what_they_leave_to_python(how):
    """The collectives of api.World as native methods: the same calls and codes as the methods written in Python."""
    class Sub(api.World):
        def all_reduce(self, *args):
            return super().all_reduce(*args)
    w = (Sub if how == "subclass" else api.World)(2, dry=True)
    assert type(api.World.__dict__["all_reduce"]).__name__ == "Method"
    for r in range(2):
        rank = bool(r) if how == "boolean rank" else r
        args = ((r + 1) << 20, (r + 10) << 20, 100, Kind.FP32 if how == "kind" else T.FP32, T.SUM, 1)
        if how == "keywords":
            names = ("send", "recv", "count", "dtype", "op", "stream")
            assert w.all_reduce(rank, **dict(zip(names, args))) == 0
        elif how == "unbound":
            assert api.World.all_reduce(w, rank, *args) == 0
        else:
            assert w.all_reduce(rank, *args) == 0
    assert w.last_info().algName
    w.close()


def test_what_a_method_refuses(world):
    args = (1 << 20, 2 << 20, 10, T.FP32, T.SUM, 1)
    for bad, kind in (((2,) + args, IndexError), ((1.5,) + args, TypeError), ((0,) + args[:-1], TypeError), ((1 << 70,) + args, IndexError)):
        with pytest.raises(kind):
            world.all_reduce(*bad)
    for table in (5, None):   # an address in the place of a table is not taken for one
        with pytest.raises(TypeError):
            world.all_gather_v(0, 1 << 20, 5, 2 << 20, table, [0, 5], T.FP32, 1)
    assert world.all_reduce(0, 1 << 20, 2 << 20, 10, 99, T.SUM, 1) != 0
    closed = api.World(2, dry=True)
    closed.close()
    with pytest.raises(IndexError):
        closed.all_reduce(0, *args)


def test_ranks_that_run_ahead(world):
    """One rank's calls wait, in order, for the other's; counts that differ are found out at their own collective."""
    counts = [3 + k % 5 for k in range(200)]
    for c in counts:
        assert world.all_to_all(0, 1 << 20, c, 10 << 20, T.FP32, 1) == 0
    for k, c in enumerate(counts):
        wrong = k in (70, 199)
        assert (world.all_to_all(1, 2 << 20, c + wrong, 11 << 20, T.FP32, 1) != 0) == wrong


@pytest.mark.parametrize("name", ["all_reduce", "reduce_scatter", "reduce_scatter_v", "all_gather", "all_gather_v", "all_to_all_v", "all_to_all",
                                  "all_to_all_vc"])
def test_a_native_method_is_a_function_to_a_program(world, name):
    """What tracing decorators, documentation tools and pickle ask of a method."""
    for m in (getattr(api.World, name), getattr(world, name)):
        assert (m.__name__, m.__qualname__, m.__module__) == (name, "World." + name, "hccl_amd.api")
        assert m.__doc__ is None and m.__code__.co_varnames[:2] == ("self", "rank")
        assert name in repr(m) and weakref.ref(m)() is m
    m = getattr(api.World, name)
    assert type(m).__name__ == "Method" and inspect.isfunction(m) and inspect.isroutine(m) and isinstance(m, types.FunctionType)
    assert name in dict(inspect.getmembers(api.World, inspect.isfunction)) and inspect.ismethod(getattr(world, name))
    assert list(inspect.signature(m).parameters)[:2] == ["self", "rank"] and "rank" in inspect.signature(getattr(world, name)).parameters
    assert pickle.loads(pickle.dumps(m)) is m and copy.copy(m) is m and copy.deepcopy(m) is m
    assert weakref.WeakMethod(getattr(world, name))() == getattr(world, name)
    assert functools.wraps(m)(lambda *a: None).__name__ == name
    m.seen = 5
    assert getattr(world, name).seen == 5
    del m.seen
    assert not hasattr(m, "seen") and not hasattr(m, "no_such_name")


PATCHED = """
from hccl_amd import api
seen = []
def traced(of):
    def call(*args, **kw):
        seen.append(of.__name__)
        return of(*args, **kw)
    return call
for name in ("all_reduce", "all_gather_v"):
    setattr(api.World, name, traced(getattr(api.World, name)))
w = api.World(2, dry=True)
for r in range(2):
    assert w.all_reduce(r, (r + 1) << 20, (r + 10) << 20, 100, 4, 0, 1) == 0
    assert w.all_gather(r, (r + 1) << 20, (r + 10) << 20, 100, 4, 1) == 0
assert seen == ["all_reduce"] * 2, seen
assert type(api.World.__dict__["all_gather"]).__name__ == "Method"
"""


def test_methods_replaced_before_the_first_communicator_stay():
    run = subprocess.run([sys.executable, "-c", PATCHED], cwd=ROOT, capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stderr[-2000:]


EMPTIED_MEANWHILE = """
import ctypes
from hccl_amd import api
w = api.World(2, dry=True)
class Table(bytearray):
    @property
    def __class__(self):
        w.comms.clear()
        return type(api.u64_table([1]))
try:
    w.reduce_scatter_v(0, 1 << 20, Table(16), Table(16), 2 << 20, 0, 4, 0, 1)   # a call of the rank it was made for, or an error
except (IndexError, TypeError):
    pass
print("ended")
"""


def test_an_argument_that_empties_the_communicators_while_it_is_looked_at():
    run = subprocess.run([sys.executable, "-c", EMPTIED_MEANWHILE], cwd=ROOT, capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and run.stdout == "ended\n", (run.returncode, run.stdout, run.stderr[-2000:])

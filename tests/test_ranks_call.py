"""The Python mirror's native loop over the ranks: what it recognises, what it leaves to ctypes, and that both ways the
library sees the same arguments (told apart by its return codes; no GPU needed: without one a complete collective ends with
HCCL_E_RUNTIME)."""
import ctypes
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest
import torch

from hccl_loader import load

H = load()
P = 4


@pytest.fixture
def comms():
    c = H.comm_init_all(P)
    yield c
    H.comm_destroy(c)


def _code(fn, *args, **kw):
    try:
        fn(*args, **kw)
    except H.HcclError as e:
        return e.code
    return 0


ISSUED = 0 if torch.cuda.is_available() else H.HCCL_E_RUNTIME


@pytest.mark.parametrize("form", [list, tuple, lambda x: iter(list(x)), lambda x: [ctypes.c_void_p(v) for v in x]])
def test_sequences_and_pointer_types(comms, form):
    if torch.cuda.is_available():
        pytest.skip("host pointers: only where no collective is issued")
    ptrs = [0x100000 * (r + 1) for r in range(P)]
    for fn in (H.all_reduce, H.reduce_scatter):
        assert _code(fn, comms, form(ptrs), form([p + 0x80000 for p in ptrs]), 16, H.HCCL_DATA_TYPE_FP32, 0, 1) == ISSUED
        # a null pointer of the second rank: its call fails, the first rank has arrived and is still waiting
        assert _code(fn, comms, [ptrs[0], None, ptrs[2], ptrs[3]], ptrs, 16, H.HCCL_DATA_TYPE_FP32, 0, 1) == H.HCCL_E_PTR
        assert _code(fn, comms, ptrs, ptrs, 16, H.HCCL_DATA_TYPE_FP32, 0, 1) == H.HCCL_E_AGAIN
        # the others join what the first rank started
        assert _code(fn, comms[1:], ptrs[1:], ptrs[1:], 16, H.HCCL_DATA_TYPE_FP32, 0, 1) == ISSUED


def test_every_kind_reaches_its_call(comms):
    a = [0x100000 * (r + 1) for r in range(P)]
    none = [None] * P
    dt = H.HCCL_DATA_TYPE_FP32
    calls = [(H.all_reduce, (none, a, 8, dt, 0, 1)), (H.reduce_scatter, (none, a, 8, dt, 0, 1)), (H.reduce_scatter_no_alloc, (none, a, 8, dt, 0, 1)),
             (H.all_gather, (none, a, 8, dt, 1)), (H.all_to_all, (none, a, 8, dt, 1)), (H.broadcast, (none, 8, dt, 0, 1)),
             (H.reduce, (none, a, 8, dt, 0, 0, 1)), (H.scatter, (a, none, 8, dt, 0, 1))]
    for fn, args in calls:
        with pytest.raises(H.HcclError) as e:
            fn(comms, *args)
        assert e.value.code == H.HCCL_E_PTR and ("Hccl" + "".join(w.title() for w in fn.__name__.split("_"))
                                                 .replace("AllToAll", "AlltoAll").replace("ReduceScatterNoAlloc", "AmdReduceScatterNoAlloc")) in str(e.value)


@pytest.mark.parametrize("kind", ["uint64", "int64", "lists", "transposed", "tables", "ctypes tables"])
def test_all_to_all_v_tables(comms, kind):
    if torch.cuda.is_available():
        pytest.skip("host pointers: only where no collective is issued")
    rng = np.random.default_rng(3)
    cnt = rng.integers(0, 9, (P, P)).astype(np.int64)
    back = np.ascontiguousarray(cnt.T)
    dis, rdis = np.cumsum(cnt, axis=1) - cnt, np.cumsum(back, axis=1) - back
    ptrs = [0x100000 * (r + 1) for r in range(P)]

    def run(c, b):
        t = [c, dis, b, rdis]
        kw = {}
        if kind == "uint64":
            t = [x.astype(np.uint64) for x in t]
        elif kind == "lists":
            t = [x.tolist() for x in t]
        elif kind == "transposed":
            t = [np.asfortranarray(x.astype(np.uint64)) for x in t]
        elif kind != "int64":
            kw["tables"] = H.a2av_tables(*([x.tolist() for x in t] if kind == "ctypes tables" else t))
            t = [None] * 4
        return _code(H.all_to_all_v, comms, ptrs, t[0], t[1], [p + 0x80000 for p in ptrs], t[2], t[3], H.HCCL_DATA_TYPE_INT32, 1, **kw)

    assert run(cnt, back) == ISSUED
    wrong = back.copy()
    wrong[2, 1] += 1                    # rank 2 expects one more from rank 1 than it sends
    assert run(cnt, wrong) == H.HCCL_E_PARA


# ---- start-up: in a process of its own, on a copy of the package beside a link to the built library ----------------

START = """
import importlib.util, sys
spec = importlib.util.spec_from_file_location("mirror", sys.argv[1])
H = importlib.util.module_from_spec(spec)
spec.loader.exec_module(H)
comms = H.comm_init_all(2)
try:
    H.all_reduce(comms, [None, None], [4096, 8192], 8, H.HCCL_DATA_TYPE_FP32, 0, 1)
except H.HcclError as e:
    print("code", e.code, "native", int(H._call is not H._through_ctypes))
"""


def _start(tmp_path, with_extension, env=None):
    package = os.path.dirname(os.path.dirname(H.LIB_PATH))
    tree = tmp_path / "tree"
    (tree / "lib").mkdir(parents=True)
    shutil.copy(os.path.join(package, "__init__.py"), tree)
    os.symlink(H.LIB_PATH, tree / "lib" / "libhccl.so")
    if with_extension == "broken":
        (tree / "lib" / os.path.basename(H.RANKS_PATH)).write_bytes(b"not a library")
    elif with_extension:
        os.symlink(H.RANKS_PATH, tree / "lib" / os.path.basename(H.RANKS_PATH))
    r = subprocess.run([sys.executable, "-c", START, str(tree / "__init__.py")], env={**os.environ, **(env or {})}, stdout=subprocess.PIPE,
                       stderr=subprocess.PIPE, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    return r.stdout.strip()


@pytest.mark.parametrize("with_extension,native", [(True, 1), (False, 0), ("broken", 0)])
def test_starts_without_the_extension(tmp_path, with_extension, native):
    # a tree that was built with another interpreter, or without its headers, holds no extension for this one
    assert _start(tmp_path, with_extension) == "code %d native %d" % (H.HCCL_E_PTR, native)


def test_the_library_called_is_the_one_loaded(tmp_path):
    # another libhccl.so on the loader's search path, every function of which fails with 77
    stub = tmp_path / "elsewhere"
    stub.mkdir()
    src = stub / "stub.cc"
    src.write_text("".join('extern "C" int %s() { return 77; }\n' % name for name in H.EXPORTS))
    subprocess.run(["g++", "-shared", "-fPIC", str(src), "-o", str(stub / "libhccl.so")], check=True)
    path = str(stub) + os.pathsep + os.environ.get("LD_LIBRARY_PATH", "")
    assert _start(tmp_path, True, {"LD_LIBRARY_PATH": path}) == "code %d native 1" % H.HCCL_E_PTR


# ---- which calls the native loop takes ------------------------------------------------------------------------------

def test_what_the_native_loop_recognises(comms):
    a = [0x100000 * (r + 1) for r in range(P)]
    none = [None] * P
    dt = H.HCCL_DATA_TYPE_FP32

    def call(comms, sends, recvs, kind=H._ALL_REDUCE, count=8, stream=1, tables=None):
        return H._call(kind, comms, sends, recvs, count, dt, 0, 0, stream, tables)

    # (null send buffers: the first rank's call fails, so that nothing is left waiting)
    for same in (list, tuple):
        for recvs in (a, [ctypes.c_void_p(v) for v in a]):
            assert call(same(comms), same(none), same(recvs)) == H.HCCL_E_PTR
    assert call(comms, none, a, stream=ctypes.c_void_p(1)) == H.HCCL_E_PTR
    for form in (iter, np.array, lambda x: dict(enumerate(x)), lambda x: [np.uint64(v) for v in x], lambda x: [ctypes.c_uint64(v) for v in x],
                 lambda x: [float(v) for v in x]):
        assert call(comms, none, form(a)) == -1, form
    assert call(comms, none, a, count=8.0) == -1 and call(comms, none, a, stream="1") == -1
    assert call([comms[0]] * 65, [None] * 65, [1] * 65) == -1

    cnt = np.ones((P, P), np.uint64)
    for good in (cnt, np.ascontiguousarray(cnt.T)):
        assert call(comms, none, a, kind=H._ALL_TO_ALL_V, tables=[good] * 4) in (H.HCCL_E_PTR, H.HCCL_E_PARA)
    for bad in (cnt.astype(np.int64), cnt.astype(np.uint32), cnt.astype(">u8"), np.ones((P, 2 * P), np.uint64)[:, ::2], np.ones((P, P + 1), np.uint64),
                np.ones(P * P, np.uint64), cnt.tolist(), None):
        assert call(comms, none, a, kind=H._ALL_TO_ALL_V, tables=(cnt, cnt, bad, cnt)) == -1, bad
    assert call(comms, none, a, kind=H._ALL_TO_ALL_V, tables=(cnt, cnt, cnt)) == -1
    assert call(comms, none, a, kind=H._ALL_TO_ALL_V) == -1

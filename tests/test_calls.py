"""The engine's calls through pegaflow_amd._calls against the ctypes packing of the
same arguments: what reaches the C function, for every form a caller may use.  The
functions called are recorders of the test's own; no library, no GPU."""

import ctypes as C
import dataclasses
import os
import shutil
import subprocess
import sys
import sysconfig
import types

import numpy as np
import pytest

from pegaflow_amd import _calls, _lib
from pegaflow_amd import engine as E

P8, P32, P64, PI64 = (C.POINTER(t) for t in (C.c_uint8, C.c_uint32, C.c_uint64, C.c_int64))
SAVE = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_char_p, C.c_uint64, C.c_uint64, C.c_int, C.POINTER(_lib.PfLayerSave),
                   C.c_uint64)
QUERY = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_char_p, C.POINTER(P8), P32, C.c_uint64, P64, P64)
LOAD = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_char_p, C.c_uint64, C.c_int, C.c_uint64, C.POINTER(C.POINTER(C.c_char_p)),
                   P64, C.c_uint64, C.POINTER(PI64), C.c_uint64, C.c_char_p, C.POINTER(C.c_void_p))
WAIT = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_int, C.POINTER(_lib.PfTaskResult))


def address(fn):
    return C.cast(fn, C.c_void_p).value


def hashes_at(ptrs, lens, n):
    return [C.string_at(ptrs[i], lens[i]) for i in range(n)]


class Bytes(bytes):
    pass


class Name(str):
    pass


HASHES = [[], [b"a"], (b"ab", b"", bytes(range(40))), [b"x" * 32] * 5]
ODD_HASHES = [[bytearray(b"ab")], [b"a", Bytes(b"b")], iter([b"a"]), [memoryview(b"abc")], np.array([b"a"]), ["a"],
              [b"a", None], None]


@pytest.mark.parametrize("hashes", HASHES + ODD_HASHES, ids=lambda h: type(h).__name__)
def test_query(hashes):
    seen = []

    def fn(engine, instance, ptrs, lens, n, hits, lease):
        seen.append((engine, instance, hashes_at(ptrs, lens, n)))
        hits[0], lease[0] = 7, 2**63 + 1
        return 0

    made = _calls.query(address(QUERY(fn)), 0x1234, "inst", hashes)
    if any(hashes is h for h in ODD_HASHES):
        assert made is None and not seen
        return
    assert made == (0, 7, 2**63 + 1)
    ptrs, lens, _keep = E._pack_hashes(hashes)
    assert seen == [(0x1234, b"inst", hashes_at(ptrs, lens, len(hashes)))] == [(0x1234, b"inst", list(hashes))]


@dataclasses.dataclass
class Odd:
    layer_name: object
    block_ids: object
    block_hashes: object


def _saves():
    ids, hashes = [4, 0, 2**64 - 1], [b"h0", b"h1", b"h2" * 20]
    return {
        "one": [E.LayerSave("l0", ids, hashes)],
        "shared": [E.LayerSave(f"läyer.{i}", ids, hashes) for i in range(40)],
        "own": tuple(E.LayerSave(f"l{i}", [i, i + 1], (b"%d" % i, b"x")) for i in range(12)),
        "mixed": [E.LayerSave("a", ids, hashes), E.LayerSave("b", (1,), [b"q"]), E.LayerSave("c", ids, hashes)],
        "empty": [],
        "no_blocks": [E.LayerSave("l", [], []), E.LayerSave("m", (), ())],
    }


def _odd_saves():
    h = [b"h"]
    return {
        "array": [E.LayerSave("l", np.array([3]), h)],
        "length": [E.LayerSave("l", [1, 2], h)],
        "negative": [E.LayerSave("l", [-1], h)],
        "large": [E.LayerSave("l", [2**64], h)],
        "bool": [E.LayerSave("l", [True], h)],
        "float": [E.LayerSave("l", [1.0], h)],
        "later": [E.LayerSave("l", [1], h), E.LayerSave("l", [None], h)],
        "name": [E.LayerSave(Name("l"), [1], h)],
        "surrogate": [E.LayerSave("\ud800", [1], h)],
        "hashes": [E.LayerSave("l", [1], [Bytes(b"h")])],
        "no_attributes": [object()],
        "generator": (s for s in _saves()["one"]),
        "packed": E.PackedSaves(_saves()["one"]),
    }


def _record_saves(seen):
    def fn(engine, instance, tp, pp, device, layers, n):
        rows = [(layers[i].layer_name, layers[i].block_ids[:layers[i].n_blocks],
                 hashes_at(layers[i].block_hashes, layers[i].block_hash_lens, layers[i].n_blocks),
                 bool(layers[i].block_ids), bool(layers[i].block_hashes), bool(layers[i].block_hash_lens))
                for i in range(n)]
        seen.append((engine, instance, tp, pp, device, rows))
        return 3
    return SAVE(fn)


@pytest.mark.parametrize("name", sorted(_saves()))
def test_save(name):
    saves, seen = _saves()[name], []
    fn = _record_saves(seen)
    assert _calls.save(address(fn), 5, "inst", 1, 2, 3, saves) == 3
    packed = E.PackedSaves(saves)
    assert fn(5, b"inst", 1, 2, 3, packed.array, packed.n) == 3
    assert seen[0] == seen[1] and len(seen[0][5]) == len(saves)


@pytest.mark.parametrize("name", sorted(_odd_saves()))
def test_saves_left_to_ctypes(name):
    seen = []
    fn = _record_saves(seen)
    assert _calls.save(address(fn), 5, "inst", 1, 2, 3, _odd_saves()[name]) is None and not seen
    assert _calls.save(address(fn), 5, "inst", np.int64(1), 2, 3, _saves()["one"]) is None and not seen


def test_saves_that_change_while_they_are_read():
    ids, hashes, seen = [1, 2], [b"a", b"b"], []

    class Grows:
        layer_name = "l"
        block_hashes = hashes

        @property
        def block_ids(self):
            saves.append(self)
            return ids

    class Empties(Grows):
        @property
        def block_ids(self):
            saves.clear()
            return ids

    fn = _record_saves(seen)
    saves = [Grows()]
    assert _calls.save(address(fn), 5, "inst", 0, 0, 0, saves) == 3 and len(seen[0][5]) == 1
    saves = [Empties(), Empties()]
    assert _calls.save(address(fn), 5, "inst", 0, 0, 0, saves) is None and len(seen) == 1


def _record_loads(seen):
    def fn(engine, instance, tp, device, groups, names, sizes, lease, dests, n, shm, task):
        seen.append((engine, instance, tp, device, [[names[g][i] for i in range(sizes[g])] for g in range(groups)],
                     lease, [dests[g][:n] for g in range(groups)], shm))
        task[0] = 0xABCDEF
        return 0
    return LOAD(fn)


@pytest.mark.parametrize("dests", [[[]], [[3]], [(3, None, 5)], [[None, None], [-7, 2**63 - 1]],
                                   [[1, 2], (3, None), [9, 9]]], ids=str)
@pytest.mark.parametrize("shm", [None, "pega_load_1"])
def test_load(dests, shm):
    groups = [["a", "lé"], ("b",), []][:len(dests)]
    seen = []
    fn = _record_loads(seen)
    assert _calls.load(address(fn), 9, "inst", 1, 2, groups, 2**64 - 3, dests, shm) == (0, 0xABCDEF)
    want = [[-1 if v is None else v for v in d] for d in dests]
    assert seen == [(9, b"inst", 1, 2, [[n.encode() for n in g] for g in groups], 2**64 - 3, want,
                     shm.encode() if shm else None)]
    for d, w in zip(dests, want):
        packed, _owner = E._pack_destinations(d)
        assert [packed[i] for i in range(len(w))] == w


@pytest.mark.parametrize("groups, dests", [
    ([], []), ([["a"]], []), ([["a"]], [[1.0]]), ([["a"]], [[True]]), ([["a"]], [np.array([1])]),
    ([["a"]], [[2**63]]), ([["a"], ["b"]], [[1], [1, 2]]), ([[Name("a")]], [[1]]), ([[b"a"]], [[1]]), (["a"], [[1]]),
    ([["a"]], [range(3)]), ([["a"]], [None])], ids=str)
def test_loads_left_to_ctypes(groups, dests):
    seen = []
    assert _calls.load(address(_record_loads(seen)), 9, "inst", 1, 2, groups, 4, dests, None) is None and not seen


@pytest.mark.parametrize("status, timeout", [(0, -1), (2, 50)])
def test_wait(status, timeout):
    seen = []

    def fn(task, timeout_ms, out):
        seen.append((task, timeout_ms))
        for i, (field, ctype) in enumerate(_lib.PfTaskResult._fields_):
            setattr(out[0], field, ctype(i + 1).value)
        out[0].paths = 5
        return status

    made = _calls.wait(address(WAIT(fn)), 77, timeout)
    r = _lib.PfTaskResult()
    assert fn(77, timeout, C.pointer(r)) == status
    assert made[0] == status and seen == [(77, timeout)] * 2
    assert E.TaskResult.from_call(*made[1:]) == E.TaskResult.from_c(r)
    assert _calls.wait(address(WAIT(fn)), 77, 1.5) is None
    assert _calls.wait(0, 77, 1) is None


def test_module_is_found_by_the_interpreter_it_was_built_for_alone(tmp_path):
    """The file carries the interpreter's tag; a package that holds one of another
    interpreter, or none, is imported without it."""
    suffix = sysconfig.get_config_var("EXT_SUFFIX")
    assert os.path.basename(_calls.__file__) == "_calls" + suffix
    package = tmp_path / "pegaflow_amd"
    package.mkdir()
    for name in os.listdir(os.path.dirname(E.__file__)):
        if name.endswith(".py"):
            shutil.copy(os.path.join(os.path.dirname(E.__file__), name), package)
    (package / "_calls.cpython-399-x86_64-linux-gnu.so").write_bytes(b"of another interpreter")
    proc = subprocess.run([sys.executable, "-c", "import pegaflow_amd.engine as e; print(e._calls)"], cwd=tmp_path,
                          capture_output=True, text=True, timeout=60, env={**os.environ, "PYTHONPATH": str(tmp_path)})
    assert proc.returncode == 0 and proc.stdout == "None\n", (proc.stdout, proc.stderr)


@pytest.mark.parametrize("native", [True, False], ids=["module", "ctypes"])
def test_calls_of_an_engine_with_and_without_the_module(native, monkeypatch):
    saves, loads, queries = [], [], []

    def query(engine, instance, ptrs, lens, n, hits, lease):
        queries.append((engine, instance, hashes_at(ptrs, lens, n)))
        hits[0], lease[0] = 2, 9
        return 0

    def wait(task, timeout_ms, out):
        assert (task, timeout_ms) == (0xABCDEF, 70)
        out[0].done, out[0].bytes, out[0].paths = 1, 4096, _lib.PF_TASK_PATH_STAGED
        return 0

    record_save = _record_saves(saves)
    lib = types.SimpleNamespace(
        pf_engine_batch_save=SAVE(lambda *a: record_save(*a) - 3), pf_engine_query_prefix=QUERY(query),
        pf_engine_batch_load=_record_loads(loads), pf_task_wait=WAIT(wait), pf_task_destroy=lambda t: 0,
        pf_engine_destroy=lambda e: 0)
    monkeypatch.setattr(E._lib, "load", lambda: lib)
    monkeypatch.setattr(E, "_addresses", {})
    if not native:
        monkeypatch.setattr(E, "_calls", None)
    eng = object.__new__(E.PegaEngine)
    eng._lib, eng.handle = lib, C.c_void_p(5)
    eng.batch_save_kv_blocks("inst", 1, 2, 3, [E.LayerSave("l0", [4, 0], [b"a", b"b"])])
    assert saves == [(5, b"inst", 1, 2, 3, [(b"l0", [4, 0], [b"a", b"b"], True, True, True)])]
    assert eng.query_prefix("inst", [b"a", b"b"]) == (2, 9) and queries == [(5, b"inst", [b"a", b"b"])]
    task = eng.batch_load_kv_blocks_multi_layer("inst", 1, 3, [["l0"]], 9, [[6, None]])
    assert loads == [(5, b"inst", 1, 3, [[b"l0"]], 9, [[6, -1]], None)]
    result = task.wait(70)
    assert (result.done, result.bytes, result.paths) == (True, 4096, ("staged",))
    task.close()
    eng.handle = None


ENDS_BESIDE_A_CALL = """
import ctypes, sys, threading, time
from pegaflow_amd import _calls

class Layer:
    layer_name, block_ids, block_hashes = "l", [1], [b"h"]
    def __del__(self, print=print):
        print("released", flush=True)

class Late:  # goes with the modules, while other threads cannot have the interpreter's lock any more
    def __del__(self, sleep=time.sleep):
        sleep(1.5)

usleep = ctypes.cast(ctypes.CDLL(None).usleep, ctypes.c_void_p).value
saves = [Layer()]
threading.Thread(target=lambda: _calls.save(usleep, 900000, "inst", 0, 0, 0, saves), daemon=True).start()
time.sleep(0.2)
saves.clear()  # the call has the last reference
sys.late = Late()
print("ending", flush=True)
"""


def test_interpreter_that_ends_beside_a_call():
    """A daemon thread inside a call is ended where it takes the interpreter's lock again:
    the objects that the call held stay, because they cannot be given back without it."""
    proc = subprocess.run([sys.executable, "-c", ENDS_BESIDE_A_CALL], capture_output=True, text=True, timeout=60,
                          cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert proc.returncode == 0 and proc.stdout == "ending\n", (proc.returncode, proc.stdout, proc.stderr)

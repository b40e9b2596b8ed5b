// Python module pegaflow_amd._calls: the engine's calls of one request (save, prefix
// query, load, wait), packed and made without ctypes.
//
// Turning the lists of a call into the arrays of the C ABI one object at a time cost
// 8 us per call and 0.1 us per block in the interpreter, a fifth of a 2 MiB load.
// The forms that every caller uses go through here: exact lists and tuples of exact
// ints, bytes and strs.  For anything else (arrays, subclasses, values out of range,
// lists of unlike length) a call returns None before it has done anything, and
// engine.py makes it its own way, with the conversions and errors it has for them.
//
// Every call takes the address of the C function to call, so the module is linked to
// nothing and a test can hand it one of its own.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cxxabi.h>

#include <cstdint>
#include <new>
#include <vector>

#include "../../../include/pegahip.h"

namespace {

PyObject* g_layer_name;    // interned attribute names
PyObject* g_block_ids;
PyObject* g_block_hashes;

// Objects that a call needs while it runs without the interpreter's lock.
class Kept {
 public:
  // A thread that wants the lock back from an interpreter that is ending is ended there
  // itself, and unwound: it does not have the lock, and its objects stay.
  ~Kept() {
    if (unlocked_) return;
    for (PyObject* o : objects_) Py_DECREF(o);
  }
  void add(PyObject* borrowed) {
    objects_.push_back(borrowed);
    Py_INCREF(borrowed);
  }
  void set_unlocked(bool unlocked) { unlocked_ = unlocked; }

 private:
  std::vector<PyObject*> objects_;
  bool unlocked_ = false;
};

bool is_sequence(PyObject* o) { return PyList_CheckExact(o) || PyTuple_CheckExact(o); }
Py_ssize_t size_of(PyObject* seq) { return PySequence_Fast_GET_SIZE(seq); }
PyObject* item(PyObject* seq, Py_ssize_t i) { return PySequence_Fast_GET_ITEM(seq, i); }

// As ctypes passes an int: the low bits.
bool integer(PyObject* o, uint64_t* out) {
  if (!PyLong_CheckExact(o)) return false;
  *out = PyLong_AsUnsignedLongLongMask(o);
  return true;
}

// UTF-8 of an exact str; the object keeps it.
const char* text(PyObject* o, Kept* kept) {
  if (!PyUnicode_CheckExact(o)) return nullptr;
  const char* s = PyUnicode_AsUTF8(o);
  if (s == nullptr) {
    PyErr_Clear();
    return nullptr;
  }
  kept->add(o);
  return s;
}

struct Hashes {
  std::vector<const uint8_t*> ptrs;
  std::vector<uint32_t> lens;
  bool pack(PyObject* seq, Kept* kept) {
    if (!is_sequence(seq)) return false;
    const Py_ssize_t n = size_of(seq);
    ptrs.assign(n ? n : 1, nullptr);
    lens.assign(n ? n : 1, 0);
    for (Py_ssize_t i = 0; i < n; ++i) {
      PyObject* h = item(seq, i);
      if (!PyBytes_CheckExact(h) || static_cast<uint64_t>(PyBytes_GET_SIZE(h)) > UINT32_MAX) return false;
      ptrs[i] = reinterpret_cast<const uint8_t*>(PyBytes_AS_STRING(h));
      lens[i] = static_cast<uint32_t>(PyBytes_GET_SIZE(h));
      kept->add(h);
    }
    return true;
  }
};

// Block ids of a save: whole numbers of 64 bits.
bool pack_ids(PyObject* seq, std::vector<uint64_t>* out) {
  if (!is_sequence(seq)) return false;
  const Py_ssize_t n = size_of(seq);
  out->assign(n ? n : 1, 0);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* v = item(seq, i);
    if (!PyLong_CheckExact(v)) return false;
    (*out)[i] = PyLong_AsUnsignedLongLong(v);
    if ((*out)[i] == UINT64_MAX && PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
  }
  return true;
}

// Destinations of a load: whole numbers, None for a block that is not loaded.
bool pack_destinations(PyObject* seq, std::vector<int64_t>* out) {
  const Py_ssize_t n = size_of(seq);
  out->assign(n ? n : 1, -1);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* v = item(seq, i);
    if (v == Py_None) continue;
    if (!PyLong_CheckExact(v)) return false;
    (*out)[i] = PyLong_AsLongLong(v);
    if ((*out)[i] == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
  }
  return true;
}

PyObject* not_here() { Py_RETURN_NONE; }

// Address, handle and the number of arguments that every call begins with.
template <typename Fn>
bool begin(PyObject* const* args, Py_ssize_t n, Py_ssize_t want, Fn* fn, void** handle) {
  uint64_t address = 0, h = 0;
  if (n != want || !integer(args[0], &address) || address == 0 || !integer(args[1], &h)) return false;
  *fn = reinterpret_cast<Fn>(address);
  *handle = reinterpret_cast<void*>(h);
  return true;
}

// Runs `call` without the interpreter's lock; false, with an error set, when it threw
// (the C functions do not, short of memory they cannot get).
template <typename Call>
bool unlocked(Kept& kept, Call call) {
  bool done = true;
  kept.set_unlocked(true);
  Py_BEGIN_ALLOW_THREADS
  try {
    call();
  } catch (const abi::__forced_unwind&) {
    throw;  // the thread is being ended
  } catch (...) {
    done = false;
  }
  Py_END_ALLOW_THREADS
  kept.set_unlocked(false);
  if (!done) PyErr_SetString(PyExc_RuntimeError, "the engine call threw an exception");
  return done;
}

// save(fn, engine, instance_id, tp_rank, pp_rank, device_id, saves) -> status or None
PyObject* save(PyObject*, PyObject* const* args, Py_ssize_t nargs) try {
  decltype(&pf_engine_batch_save) fn = nullptr;
  void* engine = nullptr;
  uint64_t tp = 0, pp = 0, device = 0;
  Kept kept;
  if (!begin(args, nargs, 7, &fn, &engine)) return not_here();
  const char* instance = text(args[2], &kept);
  PyObject* saves = args[6];
  if (!instance || !integer(args[3], &tp) || !integer(args[4], &pp) || !integer(args[5], &device) ||
      !is_sequence(saves)) {
    return not_here();
  }
  const Py_ssize_t n = size_of(saves);
  std::vector<pf_layer_save> layers(n ? n : 1);
  // Layers that pass the very same list share one packed copy.
  struct PackedIds {
    PyObject* of;
    std::vector<uint64_t> ids;
  };
  struct PackedHashes {
    PyObject* of;
    Hashes hashes;
  };
  std::vector<PackedIds> ids;
  std::vector<PackedHashes> hashes;
  ids.reserve(n);     // (pointers into the elements are taken below)
  hashes.reserve(n);
  for (Py_ssize_t i = 0; i < n; ++i) {
    // A property may run any code: nothing borrowed from `saves` is used behind it.
    if (i >= size_of(saves)) return not_here();
    PyObject* layer = item(saves, i);
    kept.add(layer);
    PyObject* attr[3] = {PyObject_GetAttr(layer, g_layer_name), nullptr, nullptr};
    if (attr[0]) attr[1] = PyObject_GetAttr(layer, g_block_ids);
    if (attr[1]) attr[2] = PyObject_GetAttr(layer, g_block_hashes);
    for (PyObject* a : attr) {
      if (a == nullptr) continue;
      kept.add(a);
      Py_DECREF(a);
    }
    if (attr[2] == nullptr) {
      PyErr_Clear();
      return not_here();
    }
    const char* name = text(attr[0], &kept);
    if (name == nullptr || !is_sequence(attr[1]) || !is_sequence(attr[2]) ||
        size_of(attr[1]) != size_of(attr[2])) {
      return not_here();
    }
    size_t a = ids.size();
    while (a-- > 0 && ids[a].of != attr[1]) {
    }
    if (a == static_cast<size_t>(-1)) {
      a = ids.size();
      ids.push_back({attr[1], {}});
      if (!pack_ids(attr[1], &ids[a].ids)) return not_here();
    }
    size_t b = hashes.size();
    while (b-- > 0 && hashes[b].of != attr[2]) {
    }
    if (b == static_cast<size_t>(-1)) {
      b = hashes.size();
      hashes.push_back({attr[2], {}});
      if (!hashes[b].hashes.pack(attr[2], &kept)) return not_here();
    }
    // A list that changed its length between two layers: the packed copies decide.
    const size_t count = static_cast<size_t>(size_of(attr[1]));
    if (ids[a].ids.size() != (count ? count : 1) || hashes[b].hashes.ptrs.size() != (count ? count : 1)) {
      return not_here();
    }
    layers[i] = {name, ids[a].ids.data(), hashes[b].hashes.ptrs.data(), hashes[b].hashes.lens.data(), count};
  }
  int status = 0;
  const bool done = unlocked(kept, [&] {
    status = fn(static_cast<pf_engine_t>(engine), instance, tp, pp, static_cast<int>(device), layers.data(),
                static_cast<uint64_t>(n));
  });
  if (!done) return nullptr;
  return PyLong_FromLong(status);
} catch (const std::bad_alloc&) {
  return PyErr_NoMemory();
}

// query(fn, engine, instance_id, hashes) -> (status, hits, lease) or None
PyObject* query(PyObject*, PyObject* const* args, Py_ssize_t nargs) try {
  decltype(&pf_engine_query_prefix) fn = nullptr;
  void* engine = nullptr;
  Kept kept;
  Hashes hashes;
  if (!begin(args, nargs, 4, &fn, &engine)) return not_here();
  const char* instance = text(args[2], &kept);
  if (!instance || !hashes.pack(args[3], &kept)) return not_here();
  const uint64_t n = static_cast<uint64_t>(size_of(args[3]));
  uint64_t hits = 0, lease = 0;
  int status = 0;
  const bool done = unlocked(kept, [&] {
    status = fn(static_cast<pf_engine_t>(engine), instance, hashes.ptrs.data(), hashes.lens.data(), n, &hits,
                &lease);
  });
  if (!done) return nullptr;
  return Py_BuildValue("iKK", status, static_cast<unsigned long long>(hits),
                       static_cast<unsigned long long>(lease));
} catch (const std::bad_alloc&) {
  return PyErr_NoMemory();
}

// load(fn, engine, instance_id, tp_rank, device_id, layer_groups, lease, destinations,
//      load_state_shm) -> (status, task) or None
PyObject* load(PyObject*, PyObject* const* args, Py_ssize_t nargs) try {
  decltype(&pf_engine_batch_load) fn = nullptr;
  void* engine = nullptr;
  uint64_t tp = 0, device = 0, lease = 0;
  Kept kept;
  if (!begin(args, nargs, 9, &fn, &engine)) return not_here();
  const char* instance = text(args[2], &kept);
  PyObject *groups = args[5], *dests = args[7];
  if (!instance || !integer(args[3], &tp) || !integer(args[4], &device) || !is_sequence(groups) ||
      !integer(args[6], &lease) || !is_sequence(dests)) {
    return not_here();
  }
  const char* shm = nullptr;
  if (args[8] != Py_None && (shm = text(args[8], &kept)) == nullptr) return not_here();
  const Py_ssize_t g = size_of(groups);
  if (g == 0 || size_of(dests) < g || !is_sequence(item(dests, 0))) return not_here();
  const Py_ssize_t n = size_of(item(dests, 0));
  std::vector<std::vector<const char*>> names(g);
  std::vector<std::vector<int64_t>> ids(g);
  std::vector<const char* const*> name_ptrs(g);
  std::vector<uint64_t> sizes(g);
  std::vector<const int64_t*> id_ptrs(g);
  for (Py_ssize_t i = 0; i < g; ++i) {
    PyObject *group = item(groups, i), *list = item(dests, i);
    if (!is_sequence(group) || !is_sequence(list) || size_of(list) != n) return not_here();
    sizes[i] = static_cast<uint64_t>(size_of(group));
    names[i].assign(sizes[i] ? sizes[i] : 1, nullptr);
    for (uint64_t k = 0; k < sizes[i]; ++k) {
      names[i][k] = text(item(group, static_cast<Py_ssize_t>(k)), &kept);
      if (names[i][k] == nullptr) return not_here();
    }
    if (!pack_destinations(list, &ids[i])) return not_here();
    name_ptrs[i] = names[i].data();
    id_ptrs[i] = ids[i].data();
  }
  pf_task_t task = nullptr;
  int status = 0;
  const bool done = unlocked(kept, [&] {
    status = fn(static_cast<pf_engine_t>(engine), instance, tp, static_cast<int>(device),
                static_cast<uint64_t>(g), name_ptrs.data(), sizes.data(), lease, id_ptrs.data(),
                static_cast<uint64_t>(n), shm, &task);
  });
  if (!done) return nullptr;
  return Py_BuildValue("iK", status, static_cast<unsigned long long>(reinterpret_cast<uintptr_t>(task)));
} catch (const std::bad_alloc&) {
  return PyErr_NoMemory();
}

// wait(fn, task, timeout_ms) -> (status, done, bytes, elapsed_ms, paths, staged_groups,
// zero_copy_launches, link_copies, phases) or None; `phases` in the order of
// TaskResult.phases_ms
PyObject* wait(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  decltype(&pf_task_wait) fn = nullptr;
  void* task = nullptr;
  uint64_t timeout = 0;
  if (!begin(args, nargs, 3, &fn, &task) || !integer(args[2], &timeout)) return not_here();
  pf_task_result r = {};
  int status = 0;
  Kept kept;
  if (!unlocked(kept, [&] { status = fn(static_cast<pf_task_t>(task), static_cast<int>(timeout), &r); })) {
    return nullptr;
  }
  return Py_BuildValue("iiKdIIII(ddddddddd)", status, r.done, static_cast<unsigned long long>(r.bytes),
                       r.elapsed_ms, r.paths, r.staged_groups, r.zero_copy_launches, r.link_copies,
                       r.resolve_ms, r.queue_ms, r.convert_ms, r.plan_ms, r.staging_alloc_ms, r.enqueue_ms,
                       r.sync_ms, r.device_first_ms, r.device_ms);
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyMethodDef method(const char* name, const char* doc) {
  return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F)), METH_FASTCALL, doc};
}

PyMethodDef g_methods[] = {
    method<save>("save", "pf_engine_batch_save of a list of LayerSave: status, or None"),
    method<query>("query", "pf_engine_query_prefix: (status, hits, lease), or None"),
    method<load>("load", "pf_engine_batch_load: (status, task), or None"),
    method<wait>("wait", "pf_task_wait: (status, fields of the result), or None"),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_calls", "Engine calls without ctypes.", -1, g_methods,
                        nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls(void) {
  g_layer_name = PyUnicode_InternFromString("layer_name");
  g_block_ids = PyUnicode_InternFromString("block_ids");
  g_block_hashes = PyUnicode_InternFromString("block_hashes");
  if (!g_layer_name || !g_block_ids || !g_block_hashes) return nullptr;
  return PyModule_Create(&g_module);
}

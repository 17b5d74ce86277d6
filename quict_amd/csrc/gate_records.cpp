// Gate objects of a circuit -> qs_gate records, in one pass over the list.
//
// A circuit of 400 gates on 20 qubits takes the GPU 0.14 ms; reading its gates
// attribute by attribute in Python took 0.4 ms, here 0.04 ms.  The fixed gate types are copied
// from one prototype record per type and precision, and Rx, Ry, Rz, CRz, U1, CU1 and U3
// get their payloads from the closed forms; everything else is left to the caller.
//
// Loaded with ctypes.PyDLL (the interpreter lock is held, Python errors pass through);
// no state is kept between calls.
#include <Python.h>

#include "../../include/qsim.h"

#include <cmath>
#include <complex>
#include <cstring>
#include <utility>
#include <vector>

namespace {

using zc = std::complex<double>;

enum Code { RX = 0, RY, RZ, CRZ, U1, CU1, U3, NROT };  // then the fixed types, two prototypes each

// One value per pointer, few of them: a small open table.
class PointerMap {
 public:
  explicit PointerMap(size_t n) {
    size_t s = 16;
    while (s < 4 * n) s *= 2;
    slots.assign(s, {nullptr, -1});
  }
  int find(const void* p) const {
    for (size_t i = at(p);; i = (i + 1) & (slots.size() - 1)) {
      if (slots[i].first == p) return slots[i].second;
      if (!slots[i].first) return -1;
    }
  }
  void add(const void* p, int v) {
    size_t i = at(p);
    while (slots[i].first) i = (i + 1) & (slots.size() - 1);
    slots[i] = {p, v};
  }

 private:
  std::vector<std::pair<const void*, int>> slots;
  size_t at(const void* p) const { return ((size_t)p >> 4) * 0x9E3779B97F4A7C15ull >> 32 & (slots.size() - 1); }
};

// The classes seen in this call, and whether they read their attributes as `base` does.
class Classes {
 public:
  explicit Classes(PyObject* b) : base(b) {}
  int plain(PyTypeObject* t) {  // -1: error
    for (const auto& c : seen)
      if (c.first == t) return c.second;
    int ok = PyType_IsSubtype(t, (PyTypeObject*)base);
    for (const char* name : {"type", "cargs", "targs", "pargs", "precision", "__getattribute__"}) {
      if (!ok) break;
      PyObject* a = PyObject_GetAttrString((PyObject*)t, name);
      PyObject* b = PyObject_GetAttrString(base, name);
      if (!a || !b) {
        Py_XDECREF(a), Py_XDECREF(b);
        return -1;
      }
      ok = a == b;
      Py_DECREF(a), Py_DECREF(b);
    }
    seen.push_back({t, ok});
    return ok;
  }

 private:
  PyObject* base;
  std::vector<std::pair<PyTypeObject*, int>> seen;
};

struct Ref {  // owned
  PyObject* p;
  explicit Ref(PyObject* o) : p(o) {}
  ~Ref() { Py_XDECREF(p); }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
};

// Payload of rotation `code`; false: a dense matrix that is diagonal after all, which
// the caller's general path turns into another kind of record.
bool rotation(int code, const double* a, bool single, qs_gate& g) {
  zc m[4];
  int n = 1;
  g.kind = QS_GATE_DENSE;
  g.ncontrols = 0;
  g.ntargets = 1;
  if (code == RX || code == RY) {
    const double c = std::cos(a[0] / 2), s = std::sin(a[0] / 2);
    n = 4;
    m[0] = m[3] = c;
    if (code == RX) m[1] = m[2] = zc(0, -s);
    else m[1] = -s, m[2] = s;
  } else if (code == U3) {
    const double c = std::cos(a[0] / 2), s = std::sin(a[0] / 2);
    n = 4;
    m[0] = c;
    m[1] = -zc(std::cos(a[2]), std::sin(a[2])) * s;
    m[2] = zc(std::cos(a[1]), std::sin(a[1])) * s;
    m[3] = zc(std::cos(a[1] + a[2]), std::sin(a[1] + a[2])) * c;
  } else if (code == U1 || code == CU1) {
    g.kind = QS_GATE_PHASE;
    g.ncontrols = code == CU1;
    m[0] = zc(std::cos(a[0]), std::sin(a[0]));
  } else {  // Rz, CRz
    g.kind = QS_GATE_DIAG;
    g.ncontrols = code == CRZ;
    n = 2;
    m[0] = zc(std::cos(a[0] / 2), -std::sin(a[0] / 2));
    m[1] = zc(std::cos(a[0] / 2), std::sin(a[0] / 2));
  }
  if (single)
    for (int i = 0; i < n; ++i) m[i] = zc((float)m[i].real(), (float)m[i].imag());
  if (n == 4 && m[1] == 0.0 && m[2] == 0.0) return false;
  if (n == 2 && m[0] == 1.0) {
    g.kind = QS_GATE_PHASE;
    m[0] = m[1], n = 1;
  }
  std::memcpy(g.m, m, n * sizeof(zc));
  return true;
}

}  // namespace

extern "C" {

// gates: list of n_gates; base: the gate class; types: tuple of the NROT rotation types,
// then the fixed types; c128, c64: the precisions; protos: records of the fixed types in
// order, each in c128 and c64; n: qubits.  Fills out[0..n_gates) except the gates that
// are left to the caller, whose numbers go to left.  Returns how many those are, or -1
// with a Python error set.
int gate_records(PyObject* gates, PyObject* base, PyObject* types, PyObject* c128, PyObject* c64, const qs_gate* protos,
                 int n, qs_gate* out, int32_t* left) {
  static PyObject* names[5];
  if (!names[0]) {
    const char* s[5] = {"_type", "_cargs", "_targs", "_pargs", "_precision"};
    for (int i = 4; i >= 0; --i)
      if (!(names[i] = PyUnicode_InternFromString(s[i]))) return -1;
  }
  if (!PyList_Check(gates) || !PyTuple_Check(types) || !PyType_Check(base)) {
    PyErr_SetString(PyExc_TypeError, "gate_records: bad arguments");
    return -1;
  }
  const Py_ssize_t G = PyList_GET_SIZE(gates), T = PyTuple_GET_SIZE(types);
  PointerMap codes((size_t)T);
  for (Py_ssize_t i = 0; i < T; ++i) codes.add(PyTuple_GET_ITEM(types, i), (int)i);
  Classes classes(base);
  int nleft = 0;
  for (Py_ssize_t k = 0; k < G; ++k) {
    if (k >= PyList_GET_SIZE(gates)) {
      PyErr_SetString(PyExc_RuntimeError, "gate list changed while it was read");
      return -1;
    }
    Ref g(PyList_GET_ITEM(gates, k));
    Py_INCREF(g.p);
    const int plain = classes.plain(Py_TYPE(g.p));
    if (plain < 0) return -1;
    if (!plain) {
      left[nleft++] = (int32_t)k;
      continue;
    }
    Ref type(PyObject_GetAttr(g.p, names[0])), ca(PyObject_GetAttr(g.p, names[1])), ta(PyObject_GetAttr(g.p, names[2])),
        prec(PyObject_GetAttr(g.p, names[4]));
    if (!type.p || !ca.p || !ta.p || !prec.p) return -1;
    const int code = codes.find(type.p);
    const bool single = prec.p == c64;
    if (code < 0 || (!single && prec.p != c128) || !PyList_Check(ca.p) || !PyList_Check(ta.p) ||
        PyList_GET_SIZE(ca.p) + PyList_GET_SIZE(ta.p) > QS_MAX_GATE_BITS) {
      left[nleft++] = (int32_t)k;
      continue;
    }
    qs_gate& r = out[k];
    if (code < NROT) {
      Ref pa(PyObject_GetAttr(g.p, names[3]));
      if (!pa.p) return -1;
      const Py_ssize_t np = code == U3 ? 3 : 1;
      if (!PyList_Check(pa.p) || PyList_GET_SIZE(pa.p) != np) {
        left[nleft++] = (int32_t)k;
        continue;
      }
      double a[3] = {0, 0, 0};
      for (Py_ssize_t i = 0; i < np; ++i) {
        a[i] = PyFloat_AsDouble(PyList_GET_ITEM(pa.p, i));
        if (a[i] == -1.0 && PyErr_Occurred()) return -1;
      }
      std::memset(&r, 0, sizeof(r));
      if (!rotation(code, a, single, r)) {
        left[nleft++] = (int32_t)k;
        continue;
      }
    } else {
      r = protos[2 * (code - NROT) + single];
    }
    int b = 0;
    for (PyObject* l : {ca.p, ta.p})
      for (Py_ssize_t i = 0; i < PyList_GET_SIZE(l); ++i) {
        const long q = PyLong_AsLong(PyList_GET_ITEM(l, i));
        if (q == -1 && PyErr_Occurred()) return -1;
        r.bits[b++] = (int32_t)(n - 1 - q);
      }
  }
  return nleft;
}

}  // extern "C"

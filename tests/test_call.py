"""The native calls of the Python binding (csrc/call.cpp) against the ctypes ones: the same arguments arrive, and what
is not of the usual types is converted or refused as ctypes does."""
import ctypes
import os
import subprocess
import sys
import sysconfig

import numpy as np
import pytest
import torch

import cumpsgemm_amd as cg
from cumpsgemm_amd import _lib

STUB = """
#include <stdint.h>
#include <string.h>
extern "C" {
double got[32];
static int put(int n, const double *v) { memcpy(got, v, n * sizeof(double)); return n; }
#define P(x) (double)(uintptr_t)(x)
#define V P(h), (double)oa, (double)ob
int sgemm(void *h, int oa, int ob, uint64_t m, uint64_t n, uint64_t k, const float *al, void *a, uint64_t lda, void *b,
          uint64_t ldb, const float *be, void *c, uint64_t ldc, int mode) {
  const double v[] = {V, (double)m, (double)n, (double)k, al[0], P(a), (double)lda, P(b), (double)ldb, be[0], P(c), (double)ldc, (double)mode};
  return put(15, v); }
int cgemm(void *h, int oa, int ob, uint64_t m, uint64_t n, uint64_t k, const float *al, void *a, uint64_t lda, void *b,
          uint64_t ldb, const float *be, void *c, uint64_t ldc, int mode) {
  const double v[] = {V, (double)m, (double)n, (double)k, al[0], al[1], P(a), (double)lda, P(b), (double)ldb, be[0], be[1], P(c), (double)ldc, (double)mode};
  return put(17, v); }
int sbatch(void *h, int oa, int ob, uint64_t m, uint64_t n, uint64_t k, const float *al, void *a, uint64_t lda, uint64_t sa,
           void *b, uint64_t ldb, uint64_t sb, const float *be, void *c, uint64_t ldc, uint64_t sc, uint64_t batch, int mode) {
  const double v[] = {V, (double)m, (double)n, (double)k, al[0], P(a), (double)lda, (double)sa, P(b), (double)ldb, (double)sb, be[0], P(c), (double)ldc, (double)sc, (double)batch, (double)mode};
  return put(19, v); }
int cbatch(void *h, int oa, int ob, uint64_t m, uint64_t n, uint64_t k, const float *al, void *a, uint64_t lda, uint64_t sa,
           void *b, uint64_t ldb, uint64_t sb, const float *be, void *c, uint64_t ldc, uint64_t sc, uint64_t batch, int mode) {
  const double v[] = {V, (double)m, (double)n, (double)k, al[0], al[1], P(a), (double)lda, (double)sa, P(b), (double)ldb, (double)sb, be[0], be[1], P(c), (double)ldc, (double)sc, (double)batch, (double)mode};
  return put(21, v); }
int spipe(void *h, int oa, int ob, uint64_t m, uint64_t n, uint64_t k, const float *al, void *a, uint64_t lda, uint64_t sa,
          void *b, uint64_t ldb, uint64_t sb, const float *be, void *c, uint64_t ldc, uint64_t sc, uint64_t batch, int mode,
          int restore, unsigned *ids) {
  ids[0] = 7; ids[1] = 8; ids[2] = 9u + restore;
  return sbatch(h, oa, ob, m, n, k, al, a, lda, sa, b, ldb, sb, be, c, ldc, sc, batch, mode); }
int cpipe(void *h, int oa, int ob, uint64_t m, uint64_t n, uint64_t k, const float *al, void *a, uint64_t lda, uint64_t sa,
          void *b, uint64_t ldb, uint64_t sb, const float *be, void *c, uint64_t ldc, uint64_t sc, uint64_t batch, int mode,
          int restore, unsigned *ids) {
  ids[0] = 7; ids[1] = 8; ids[2] = 9u + restore;
  return cbatch(h, oa, ob, m, n, k, al, a, lda, sa, b, ldb, sb, be, c, ldc, sc, batch, mode); }
int s2x2(void *h, int oa, int ob, uint64_t m, const float *al, void *a, uint64_t lda, uint64_t sa, void *b, uint64_t ldb,
         uint64_t sb, const float *be, void *c, uint64_t ldc, uint64_t sc, uint64_t batch) {
  return sbatch(h, oa, ob, m, 0, 0, al, a, lda, sa, b, ldb, sb, be, c, ldc, sc, batch, 0); }
int c2x2(void *h, int oa, int ob, uint64_t m, const float *al, void *a, uint64_t lda, uint64_t sa, void *b, uint64_t ldb,
         uint64_t sb, const float *be, void *c, uint64_t ldc, uint64_t sc, uint64_t batch) {
  return cbatch(h, oa, ob, m, 0, 0, al, a, lda, sa, b, ldb, sb, be, c, ldc, sc, batch, 0); }
}
"""
NAMES = ("sgemm", "cgemm", "sbatch", "cbatch", "spipe", "cpipe", "s2x2", "c2x2", "s2x2", "c2x2")


@pytest.fixture
def calls(tmp_path):
    """(handle without a library behind it, the arguments its last call passed)"""
    assert _lib.lib() is not None and _lib._native is not None, "csrc/call.cpp is not built"
    (tmp_path / "stub.cpp").write_text(STUB)
    so = tmp_path / "stub.so"
    subprocess.check_call(["g++", "-shared", "-fPIC", "-o", str(so), str(tmp_path / "stub.cpp")])
    stub = ctypes.CDLL(str(so))
    address = [ctypes.cast(getattr(stub, n), ctypes.c_void_p).value for n in NAMES]
    real = [ctypes.cast(getattr(_lib.lib(), n), ctypes.c_void_p).value for n in _lib._CALL_FUNCTIONS]
    h = cg.Handle.__new__(cg.Handle)
    h._L, h._h, h._addr = _lib.lib(), None, 0x1230
    got = (ctypes.c_double * 32).in_dll(stub, "got")
    _lib._native.bind(*address)
    yield h, got
    _lib._native.bind(*real)


@pytest.mark.parametrize("cplx", [False, True])
def test_every_argument_arrives_in_its_place(calls, cplx):
    h, got = calls
    a, b, c = torch.zeros(4), torch.zeros(4), torch.zeros(4)
    pa, pb, pc = a.data_ptr(), b.data_ptr(), c.data_ptr()
    al, be = (2.5 - 1.5j, 0.5 + 0.25j) if cplx else (2.5, 0.5)
    sc = [2.5, -1.5] if cplx else [2.5], [0.5, 0.25] if cplx else [0.5]
    st = h.gemm(111, 112, 3, 4, 5, al, a, 6, pb, 7, be, c, 8, 1, cplx=cplx)
    assert list(got)[:st] == [0x1230, 111, 112, 3, 4, 5, *sc[0], pa, 6, pb, 7, *sc[1], pc, 8, 1]
    batch = [*sc[0], pa, 6, 60, pb, 7, 70, *sc[1], pc, 8, 80]
    st = h.gemm_strided_batch(111, 112, 3, 4, 5, al, a, 6, 60, b, 7, 70, be, c, 8, 80, 9, 2, cplx=cplx)
    assert list(got)[:st] == [0x1230, 111, 112, 3, 4, 5, *batch, 9, 2]
    st, ids = h.gemm_pipeline(111, 112, 3, 4, 5, al, a, 6, b, 7, be, c, 8, 9, cplx=cplx, stridea=60, strideb=70, stridec=80,
                              batch=9, restore_ab=True)
    assert list(got)[:st] == [0x1230, 111, 112, 3, 4, 5, *batch, 9, 9] and ids == (7, 8, 10)
    for f in (h.gemm_Mx2x2, h.gemm_2xNx2):
        st = f(111, 112, 3, al, a, 6, b, 7, be, c, 8, cplx=cplx, stridea=60, strideb=70, stridec=80, batch=9)
        assert list(got)[:st] == [0x1230, 111, 112, 3, 0, 0, *batch, 9, 0]
    # a real scalar of a complex product; a null pointer
    st = h.gemm(111, 112, 3, 4, 5, 1.0, None, 6, b, 7, 0.0, c, 8, 1, cplx=cplx)
    assert list(got)[6:st] == [1, *[0] * cplx, 0, 6, pb, 7, 0, *[0] * cplx, pc, 8, 1]


class Pointer:
    def data_ptr(self):
        raise ValueError("gone")


@pytest.mark.parametrize("where,value", [
    (2, np.int64(3)), (2, 3.0), (2, "3"), (2, -1), (2, 1 << 70), (0, np.int32(111)), (0, True), (5, 1), (5, np.float32(1)),
    (5, 1j), (5, "x"), (5, None), (5, torch.tensor(1.0)), (6, 0), (6, np.zeros(4)), (6, Pointer()), (6, "a"), (13, 1.0), (13, np.int64(1))])
def test_other_types_are_what_ctypes_makes_of_them(monkeypatch, where, value):
    """Without a handle the library itself refuses the call: status 3 from either side, or the exception of ctypes."""
    _lib.lib()
    h = cg.Handle.__new__(cg.Handle)
    h._L, h._h, h._addr = _lib.lib(), None, None
    args = [111, 111, 2, 2, 2, 1.0, 16, 2, 16, 2, 0.0, 16, 2, 1]
    args[where] = value

    def outcome():
        try:
            return h.gemm(*args)
        except Exception as e:  # noqa: BLE001
            return type(e)
    native = outcome()
    monkeypatch.setattr(_lib, "_native", None)
    assert native == outcome()


SEEN = """
#include <stdint.h>
#include <string.h>
extern "C" {
uint64_t seen[20];
static uint64_t bits(const float *p) { uint32_t b; memcpy(&b, p, 4); return b; }
#define ARGS void *h, int oa, int ob, uint64_t m, uint64_t n, uint64_t k, const float *al, void *a, uint64_t lda, void *b, \
  uint64_t ldb, const float *be, void *c, uint64_t ldc, int mode
#define PASS h, oa, ob, m, n, k, al, a, lda, b, ldb, be, c, ldc, mode
#define U(x) (uint64_t)(uintptr_t)(x)
static int put(int cplx, ARGS) {
  const uint64_t v[17] = {U(h), (uint32_t)oa, (uint32_t)ob, m, n, k, bits(al), U(a), lda, U(b), ldb, bits(be), U(c), ldc,
                          (uint32_t)mode, cplx ? bits(al + 1) : 0, cplx ? bits(be + 1) : 0};
  memcpy(seen, v, sizeof v);
  return 0; }
int s(ARGS) { return put(0, PASS); }
int c(ARGS) { return put(1, PASS); }
int s_ex(ARGS, unsigned *) { return put(0, PASS); }
int c_ex(ARGS, unsigned *) { return put(1, PASS); }
}
"""


@pytest.fixture(scope="module")
def seen_stub(tmp_path_factory):
    d = tmp_path_factory.mktemp("seen")
    (d / "seen.cpp").write_text(SEEN)
    subprocess.check_call(["g++", "-shared", "-fPIC", "-o", str(d / "seen.so"), str(d / "seen.cpp")])
    return ctypes.CDLL(str(d / "seen.so"))


@pytest.fixture
def seen(seen_stub):
    """(handle, what the last call passed, to the last bit): both routes end in the same functions"""
    assert _lib.lib() is not None and _lib._native is not None, "csrc/call.cpp is not built"
    stub = seen_stub
    address = [ctypes.cast(stub.s if i % 2 == 0 else stub.c, ctypes.c_void_p).value for i in range(len(NAMES))]
    real = [ctypes.cast(getattr(_lib.lib(), n), ctypes.c_void_p).value for n in _lib._CALL_FUNCTIONS]

    class Library:
        cuMpSGEMM_sgemm_ex, cuMpSGEMM_cgemm_ex = stub.s_ex, stub.c_ex
    for name in ("cuMpSGEMM_sgemm_ex", "cuMpSGEMM_cgemm_ex"):
        getattr(Library, name).argtypes = getattr(_lib.lib(), name).argtypes
        assert getattr(Library, name).argtypes, name
    h = cg.Handle.__new__(cg.Handle)
    h._L, h._h, h._addr = Library, ctypes.c_void_p(0x1230), 0x1230
    h.close = lambda: None
    _lib._native.bind(*address)
    yield h, (ctypes.c_uint64 * 20).in_dll(stub, "seen")
    _lib._native.bind(*real)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("where,value", [
    (2, np.int64(3)), (2, 3.0), (2, "3"), (2, -1), (2, 1 << 63), (2, 1 << 70), (2, (1 << 70) + 5), (2, True), (2, None),
    (0, np.int32(111)), (0, True), (0, -1), (0, 1 << 40), (0, (1 << 40) + 112), (0, (1 << 31) + 7),
    (5, 1), (5, np.float32(1)), (5, np.float64(2.5)), (5, 1j), (5, 1e300), (5, -1e-300), (5, float("nan")), (5, float("inf")),
    (5, -0.0), (5, "x"), (5, "2"), (5, None), (5, True), (5, torch.tensor(1.5)), (10, 3), (10, 2.5 - 1e300j),
    (6, 0), (6, None), (6, -1), (6, 1 << 63), (6, (1 << 70) + 16), (6, True), (6, np.int64(64)), (6, np.zeros(4)),
    (6, Pointer()), (6, "a"), (6, "32"), (6, 48.7), (11, torch.zeros(3)), (11, torch.zeros(0)),
    (13, 1.0), (13, "9"), (13, np.int64(1)), (13, -1), (13, (1 << 32) + 9), (13, None)])
def test_what_arrives_is_what_ctypes_passes(seen, monkeypatch, cplx, where, value):
    """To the last bit, or the same exception: sizes and pointers beyond 64 bits, scalars beyond FP32, other types."""
    h, got = seen
    args = [111, 112, 2, 3, 4, 1.0, 16, 5, 24, 6, 0.0, 32, 7, 1]
    args[where] = value

    def outcome():
        got[:] = [77] * 20
        try:
            return h.gemm(*args, cplx=cplx), list(got)
        except Exception as e:  # noqa: BLE001
            return type(e), list(got)
    native = outcome()
    monkeypatch.setattr(_lib, "_native", None)
    assert native == outcome()
    assert isinstance(native[0], type) or native[1][0] == 0x1230


def test_usual_arguments_do_not_go_through_ctypes(seen):
    h, got = seen
    h = type("Native", (), {"_L": None, "_h": None, "_addr": h._addr, "gemm": cg.Handle.gemm})()
    for pointer in (16, None, torch.zeros(1)):
        got[0] = 0
        assert h.gemm(111, 112, 2, 3, 4, 1.0, pointer, 5, 24, 6, 0.0, 32, 7, 1) == 0 and got[0] == 0x1230


@pytest.mark.parametrize("raised", [KeyboardInterrupt, MemoryError, ValueError])
@pytest.mark.parametrize("where", [6, 8, 11])
def test_what_a_pointer_raises_ends_the_call(calls, where, raised):
    """An interrupt that arrives inside data_ptr() is not lost, and the object is not asked again."""
    h, got = calls
    asked = []

    class Once:
        def data_ptr(self):
            asked.append(1)
            if len(asked) == 1:
                raise raised
            return 16
    args = [111, 111, 2, 2, 2, 1.0, 16, 2, 16, 2, 0.0, 16, 2, 1]
    args[where] = Once()
    got[0] = 0
    with pytest.raises(raised):
        h.gemm(*args)
    assert len(asked) == 1 and got[0] == 0


CSRC = os.path.join(os.path.dirname(os.path.abspath(_lib.__file__)), "csrc")


def _commands(*variables, **env):
    """What `make -B` would run."""
    return subprocess.run(["make", "-n", "-B", "-C", CSRC, *variables], check=True, capture_output=True, text=True,
                          env=dict(os.environ, **env)).stdout


def test_the_library_builds_without_pythons_headers(tmp_path):
    """C and C++ programs do not need call.cpp; where it cannot be compiled nothing asks for it."""
    fake = tmp_path / "python3"
    fake.write_text(f"#!/bin/sh\necho {tmp_path}\n")
    fake.chmod(0o755)
    without = _commands(PATH=f"{tmp_path}:{os.environ['PATH']}")
    assert "call.cpp" not in without and "libcumpsgemm.so" in without and "libcumpsgemm_rule.so" in without
    assert "call.cpp" in _commands()


def test_the_calls_are_built_for_one_interpreter(tmp_path, monkeypatch):
    """The one that asks, under its own suffix: another version finds no module and goes through ctypes."""
    suffix = sysconfig.get_config_var("EXT_SUFFIX")
    assert suffix != ".so"
    assert _lib.lib() is not None and _lib._native.__file__.endswith("_call" + suffix)
    other = tmp_path / "python4"
    other.write_text(f"#!{sys.executable}\nimport sys, sysconfig\nv = sysconfig.get_config_var\n"
                     "sysconfig.get_config_var = lambda n: '.cpython-400.so' if n == 'EXT_SUFFIX' else v(n)\n"
                     "exec(sys.argv[2])\n")
    other.chmod(0o755)
    assert f"/_call.cpython-400.so {CSRC}/call.cpp" in _commands(f"PYTHON={other}")
    assert f"/_call{suffix} {CSRC}/call.cpp" in _commands(f"PYTHON={sys.executable}")
    ran = []
    monkeypatch.setattr(_lib.subprocess, "check_call", ran.append)
    _lib.build()
    assert f"PYTHON={sys.executable}" in ran[0]

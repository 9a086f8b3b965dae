"""The host runtime's error paths on the CPU: the runtime's sources linked
against a HIP whose allocations and launches are made to fail on request.
Launches do nothing but check that every buffer they are given is allocated
(on a GPU, one that is not would be a memory fault) and note their order."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gturbo_amd", "csrc")

SHIM = r"""
#include <hip/hip_runtime.h>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include "gt_internal.hpp"
static std::map<const char*, size_t> live;
static std::string log_, fail_name;
static int bad = 0, fail_in = 0;  // allocations until one fails (0: none)
static int outside = 0;           // what a look for modes outside the rectangle finds
static bool dies() { return fail_in > 0 && --fail_in == 0; }
static hipError_t get(void** p, size_t n) {
  *p = nullptr;
  if (dies()) return hipErrorOutOfMemory;
  *p = calloc(1, n ? n : 1);
  live[(char*)*p] = n;
  return hipSuccess;
}
static hipError_t drop(void* p) {
  if (p && !live.erase((char*)p)) ++bad;
  free(p);
  return hipSuccess;
}
static bool ok(const void* q) {
  const char* p = (const char*)q;
  auto it = live.upper_bound(p);
  const bool in = p && it != live.begin() && (--it, p < it->first + it->second);
  bad += !in;
  return in;
}
static bool may(const void* q) { return !q || ok(q); }
static hipError_t ran(const char* name, std::initializer_list<const void*> ps) {
  for (const void* p : ps) ok(p);
  log_ += std::string(name) + " ";
  if (fail_name != name) return hipSuccess;
  fail_name.clear();
  return hipErrorLaunchFailure;
}
extern "C" {
void shim_reset() { log_.clear(); fail_name.clear(); bad = fail_in = outside = 0; }
void shim_outside(int v) { outside = v; }
void shim_fail_alloc(int k) { fail_in = k; }
void shim_fail_launch(const char* n) { fail_name = n; }
const char* shim_log() { return log_.c_str(); }
int shim_bad() { return bad; }
void* shim_device(int n) { void* p; return get(&p, n) == hipSuccess ? p : nullptr; }
hipError_t hipMalloc(void** p, size_t n) { return get(p, n); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return get(p, n); }
hipError_t hipFree(void* p) { return drop(p); }
hipError_t hipHostFree(void* p) { return drop(p); }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
  *d = nullptr;
  if (dies()) return hipErrorInvalidValue;
  *d = h;
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) {
  bool in = true;
  if (k == hipMemcpyHostToDevice || k == hipMemcpyDeviceToDevice) in = ok(d) && in;
  if (k == hipMemcpyDeviceToHost || k == hipMemcpyDeviceToDevice) in = ok(s) && in;
  if (in) memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
  return hipMemcpy(d, s, n, k);
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  if (ok(d)) memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = *t = 0; return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "made to fail"; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = nullptr; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *e = (hipGraphExec_t)malloc(1);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { free((void*)e); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = (hipEvent_t)malloc(1);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { free((void*)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { log_ += "event "; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t) { *t = 1.f; return hipSuccess; }
int roctxRangePushA(const char*) { return 0; }
int roctxRangePop() { return 0; }
}
namespace gt {
static double scratch[6 * 4097 + 6];
hipError_t glob_scratch(double** p, size_t* n) {
  live[(char*)scratch] = sizeof scratch;
  *p = scratch;
  *n = 6 * 4097 + 6;
  return hipSuccess;
}
static hipError_t y_pass(const char* name, const PassArgs& a, int mode) {
  may(a.sst);
  may(a.ka);
  may(a.fcs);
  may(a.fce);
  may(a.fph);
  if (mode == C_NLT) ok(a.out);
  else if (mode != C_START) ok(a.emk);
  if (mode == C_RK4_1 || mode == C_RK4_2 || mode == C_RK4_3 || mode == C_RK4_4 ||
      mode == C_RK4_4S)
    ok(a.znew);
  if (a.ph.akind != 1) ok(a.ka);
  if (a.fcs) { ok(a.fce); ok(a.fph); }
  return ran(name, {a.tw, a.y1, a.y2, a.z});
}
hipError_t launch_c_pass(int, int m, const PassArgs& a, hipStream_t) { return y_pass("y", a, m); }
hipError_t launch_r_pass(int, const PassArgs& a, hipStream_t) {
  return ran("x", {a.tw, a.y1, a.y2});
}
hipError_t launch_io(int, const IoArgs& a, hipStream_t) {
  log_ += a.rc.kx == a.ph.n / 2 ? "full:" : "kept:";
  if (a.mark && ok(a.mark)) *a.mark = kIoMark;
  if (a.dual) ok(a.dual);
  return ran(a.dual ? "io+ref" : "io", {a.ref, a.tw, a.y, a.cmp});
}
hipError_t launch_j_pass(int, int, const AdjArgs& a, hipStream_t) {
  may(a.snext);
  return ran("j", {a.tw, a.y1, a.y2, a.lam, a.lacc, a.emk});
}
hipError_t launch_jr_pass(int, const AdjArgs& a, hipStream_t) {
  return ran("jr", {a.tw, a.y1, a.y2});
}
hipError_t launch_produ(int, const double* z, double* u, double* v, hipStream_t) {
  return ran("produ", {z, u, v});
}
hipError_t launch_trunc_cmp(const Phys&, const Rect&, int, double2* z, hipStream_t) {
  return ran("trunc", {z});
}
hipError_t launch_gather(const Phys&, const Rect&, int, const double* r, double2* c, int, int* f,
                         hipStream_t) {
  if (f && ok(f)) *f = outside;
  return ran("gather", {r, c});
}
hipError_t launch_narrow(const Phys&, const Rect&, int, const double2* s, const Rect&, int,
                         double2* d, int, int* f, hipStream_t) {
  if (f && ok(f)) *f = outside;
  return ran("narrow", {s, d});
}
hipError_t launch_scatter(const Phys&, const Rect&, int, const double2* c, double* r,
                          hipStream_t) {
  return ran("scatter", {c, r});
}
hipError_t launch_scatter_marked(const Phys&, const Rect&, int, const double2* c, double* r,
                                 hipStream_t) {
  unsigned long long w;
  memcpy(&w, r, sizeof w);
  return w == kIoMark ? ran("scatter", {c, r}) : ran("keep", {r});
}
hipError_t launch_forcing(const Phys&, int, const ForcedMode* m, const double2* p, double,
                          double2* z, hipStream_t) {
  return ran("forcing", {m, p, z});
}
hipError_t launch_spectrum(const DiagArgs& d, int which, hipStream_t) {
  if (which) ok(d.znl);
  return ran("spectrum", {d.z, d.part1, d.part2, d.lohi, d.out1, d.out2});
}
hipError_t launch_glob(const DiagArgs& d, hipStream_t) {
  return ran("glob", {d.z, d.gpart, d.gout});
}
hipError_t launch_shell_index(const Phys&, int* ib, hipStream_t) { return ran("shell", {ib}); }
hipError_t launch_ens_c_pass(int, int, int, const PassArgs* d, const uint32_t* it, int n, int,
                             hipStream_t) {
  return ran("ens y", {d, it, it + n - 1});
}
hipError_t launch_ens_r_pass(int, int, int, const PassArgs* d, const uint32_t* it, int n, int,
                             hipStream_t) {
  return ran("ens x", {d, it, it + n - 1});
}
hipError_t launch_ens_forcing(const EnsForce* f, int, int, const int* s, hipStream_t) {
  return ran("ens forcing", {f, s});
}
hipError_t launch_ens_tick(int* s, hipStream_t) { return ran("tick", {s}); }
hipError_t launch_ka_table(const Phys&, const Rect&, int, double* k, hipStream_t) {
  return ran("ka", {k});
}
}  // namespace gt
"""

N = 1024  # (up to 512 the 2D transforms read and write reference layouts themselves)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("host")
    (d / "shim.cpp").write_text(SHIM)
    srcs = [str(d / "shim.cpp")] + [os.path.join(CSRC, f"gturbo_{s}.cpp")
                                    for s in ("runtime", "adjoint", "ensemble", "phases")]
    out = str(d / "host.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-pthread", "-D__HIP_PLATFORM_AMD__",
                    "-Wno-unused-result", "-Wl,-Bsymbolic", f"-I{CSRC}",
                    f"-I{os.path.join(ROOT, 'include')}", "-I/opt/rocm/include", *srcs, "-o", out],
                   check=True)
    L = C.CDLL(out)
    L.shim_log.restype = C.c_char_p
    L.shim_device.restype = C.c_void_p
    return L


def _params(alpv):
    return [2 * np.pi, 2 * np.pi, 1e-9, 4.0, 0.1, 0.0, alpv, 1e-3, 4, 1, 1, 1, 2.0 / 3.0, 1, 1.0,
            2.0, 4.0]


class Run:
    """A context and named arrays on that HIP; every call gives its code."""

    def __init__(self, lib, n=N):
        self.L, self.n = lib, n
        lib.shim_reset()
        self.h = C.c_void_p()
        self.a = {}
        self.out = np.zeros(2 * n)
        assert lib.gt_create(n, (C.c_double * 17)(*_params(2.0)), C.byref(self.h)) == 0

    def __call__(self, name, *args):
        return getattr(self.L, "gt_" + name)(self.h, *[self.ptr(x) for x in args])

    def ptr(self, x):
        if not isinstance(x, str):
            return x
        if x not in self.a:
            self.a[x] = np.zeros((self.n, self.n + 2))
        return C.c_void_p(self.a[x].ctypes.data)

    def enter(self, *names):
        return [self("enter_data", n, C.c_int64(self.n * (self.n + 2) * 8), 1) for n in names]

    def map(self, name):
        n = self.n * (self.n + 2) * 8
        self.dev = self.L.shim_device(n)
        return self("map_data", name, C.c_void_p(self.dev), C.c_int64(n))

    def log(self):
        return self.L.shim_log().decode().split()

    def diag(self, name, *args):
        o = self.out.ctypes.data
        two = [C.c_void_p(o), C.c_void_p(o + 8 * self.n)][:1 if name == "glob" else 2]
        return self(name, *args, *two)

    def close(self):
        self.L.gt_destroy(self.h)
        return self.L.shim_bad()


D2Z, Z2D = 1, 2


@pytest.mark.parametrize("what,fails", [("fft_dir", "allocation"), ("fft_dir", "launch"),
                                        ("copy", "allocation"), ("step4", "allocation"),
                                        ("step4", "launch")])
def test_failed_growth_of_a_compact_copy(lib, what, fails):
    """A compact copy that is to be replaced by a larger one is gone when that
    fails: what comes next reads the reference copy, or is refused where there
    is none; the array can be given back and used again."""
    r = Run(lib)
    assert r.enter("z", "w", "a", "b", "c") == [0] * 5
    assert r("trunc", "z") == 0  # z: the kept rectangle alone
    lib.shim_outside(1)
    assert r("step4", "w", "a", "c", "b", "b") == 0  # w: the whole half-spectrum
    assert r("synchronize") == 0
    if fails == "allocation":
        lib.shim_fail_alloc(1)
    else:
        lib.shim_fail_launch(b"io" if what == "fft_dir" else b"y")
    assert 0 != (r("fft_dir", "z", D2Z) if what == "fft_dir" else r("copy", "z", "w")
                 if what == "copy" else r("step4", "w", "a", "z", "b", "c"))
    n = len(r.log())
    rc = r.diag("spectrum", "z")
    if what == "fft_dir":  # its input is still there
        assert rc == 0 and r.log()[n:] == ["gather", "gather", "spectrum"]
        assert r("fft_dir", "z", D2Z) == 0
    else:
        assert rc != 0 and r.log()[n:] == [] and r("update_host", "z") != 0
        assert r("copy", "z", "w") == 0 and r("update_host", "z") == 0
    assert r("exit_data", "z", 0) == 0
    assert r.close() == 0


def test_unmapping_what_a_failed_copy_left(lib):
    """A mapped array that holds nothing after a failed copy can be unmapped."""
    r = Run(lib)
    assert r.enter("w") == [0]
    lib.shim_outside(1)
    assert r.diag("spectrum", "w") == 0
    assert r.map("z") == 0
    assert r("trunc", "z") == 0
    lib.shim_fail_alloc(1)
    assert r("copy", "z", "w") != 0 and r("update_host", "z") != 0
    assert r("unmap_data", "z") == 0
    assert r.close() == 0


@pytest.mark.parametrize("k", [1, 2, 3])
def test_failed_allocation_of_the_diagnostics(lib, k):
    """Result buffer, its device address, partial sums: whichever fails, the
    next diagnostic call allocates what is missing."""
    r = Run(lib)
    assert r.enter("z") == [0] and r("trunc", "z") == 0
    lib.shim_fail_alloc(k)
    assert r.diag("glob", "z") != 0
    assert r.diag("glob", "z") == 0 and r.diag("spectrum", "z") == 0
    assert r.close() == 0


@pytest.mark.parametrize("call", ["forced steps", "gradient"])
def test_every_allocation_may_fail(lib, call):
    """Each allocation of the calls in turn fails; the same calls again then
    succeed, on buffers that are all there."""
    for k in range(1, 100):
        r = Run(lib)
        assert r.enter("z", "w", "a", "b", "c") == [0] * 5
        seed = C.c_int32(5)

        def calls():
            if call == "gradient":
                return [r("adj_forward", "z", "w", 3, 2, C.byref(seed)),
                        r("adj_backward", "w", "a")]
            return [r("step4", "z", "a", "w", "b", "c"), r("forcing", "z", C.byref(seed)),
                    r("step4", "z", "a", "w", "b", "c"), r("fft_inv", "z", Z2D)]

        lib.shim_fail_alloc(k)
        failed = any(calls())
        assert lib.shim_bad() == 0
        lib.shim_fail_alloc(0)
        r("update_device", "z")
        assert not any(calls())
        assert r.close() == 0
        if not failed:
            break
    assert 5 < k < 99


@pytest.mark.parametrize("n", [32, N])
@pytest.mark.parametrize("array", ["host", "mapped", "mapped, a new frame"])
def test_what_an_owner_may_have_written(lib, array, n):
    """An array that was transformed and transformed again: its spectrum, unless
    the owner of a mapped one has put something else into it.  What gt_sync_ref
    gives of a mapped one is read again, too; a host array, which only
    gt_update_device changes, keeps to the compact copy."""
    r = Run(lib, n)
    host = array == "host"
    assert (r.enter("z") == [0]) if host else (r.map("z") == 0)
    assert r("fft_dir", "z", D2Z) == 0 and r.diag("spectrum", "z") == 0
    if "frame" in array:
        C.memset(C.c_void_p(r.dev), 1, 64)
    k = len(r.log())
    assert r("fft_dir", "z", D2Z) == 0
    if n == N or host:  # a mapped array's small spectrum is in its memory already
        assert r.log()[k] == ("keep" if "frame" in array else "scatter")
    assert r.log()[-1] == ("full:io" if n == N or host else "full:io+ref")
    assert r("sync_ref", "z") == 0
    k = len(r.log())
    assert r.diag("spectrum", "z") == 0
    assert ("gather" in r.log()[k:]) != host
    assert r.close() == 0


@pytest.mark.parametrize("n", [32, N])
@pytest.mark.parametrize("owned", [True, False])
def test_fft_inv_of_a_field_with_both_copies(lib, owned, n):
    """A host array's compact copy is transformed as it is, in its own size; the
    memory of a mapped one, which its owner may have written to, is read."""
    r = Run(lib, n)
    assert (r.enter("z") == [0]) if owned else (r.map("z") == 0)
    assert r("trunc", "z") == 0 and r("sync_ref", "z") == 0
    k = len(r.log())
    assert r("fft_inv", "z", Z2D) == 0
    assert r.log()[k:] == (["kept:io"] if owned else ["full:io"] if n < N
                           else ["gather", "full:io"])
    assert r.close() == 0


def test_copy_of_a_transformed_array(lib):
    """One transfer, whether or not the memory holds the spectrum, too; the copy
    has no part in what the source's owner may write."""
    for n in (32, N):
        r = Run(lib, n)
        assert r.map("z") == 0 and r.enter("w") == [0]
        assert r("fft_dir", "z", D2Z) == 0 and r("copy", "w", "z") == 0
        k = len(r.log())
        assert r("sync_ref", "w") == 0 and r.log()[k:] == ["scatter"]
        assert r.diag("spectrum", "w") == 0 and r.log()[-2:] == ["narrow", "spectrum"]
        assert r.close() == 0


@pytest.mark.parametrize("call,launches", [("fft_dir", ["full:io"]), ("trunc", ["narrow"]),
                                           ("fft_inv", ["gather", "full:io"])])
def test_timed_launches(lib, call, launches):
    """Every launch of a transform or of trunc lies inside one timed interval."""
    r = Run(lib)
    assert r.map("z") == 0
    if call == "trunc":
        assert r("fft_dir", "z", D2Z) == 0
    assert r("timing_enable", 1) == 0
    n = len(r.log())
    assert r(call, "z", *{"fft_dir": [D2Z], "trunc": [], "fft_inv": [Z2D]}[call]) == 0
    assert r.log()[n:] == ["event", *launches, "event"]
    count = (C.c_int32 * 16)()
    assert r("timing_read", None, count) == 0 and sum(count) == 1
    assert r.close() == 0


def test_failed_look_outside_the_kept_rectangle(lib):
    """A launch that fails while a transformed field is looked at for modes
    outside the kept rectangle: the next call looks again."""
    r = Run(lib)
    assert r.enter("z") == [0] and r("fft_dir", "z", D2Z) == 0
    lib.shim_fail_launch(b"narrow")
    assert r.diag("spectrum", "z") != 0
    n = len(r.log())
    assert r.diag("spectrum", "z") == 0 and r.log()[n:] == ["narrow", "spectrum"]
    assert r.close() == 0


def test_allocations_of_an_ensemble_may_fail(lib):
    """Each allocation of an ensemble's making and of a schedule with more work
    items fails in turn: no ensemble, or one that still runs the schedule it
    had."""
    n = (C.c_int32 * 2)(128, 256)
    p = (C.c_double * 34)(*_params(2.0), *_params(1.0))
    wide = (C.c_int32 * 6)(256, 256, 0, 0, 0, 1)
    for k in range(1, 100):
        lib.shim_reset()
        e = C.c_void_p()
        lib.shim_fail_alloc(k)
        rc = lib.gt_ens_create(2, n, p, C.byref(e))
        if rc != 0:
            assert not e.value and lib.shim_bad() == 0
            continue
        assert lib.gt_ens_run(e, 3) == 0
        rc = lib.gt_ens_schedule(e, wide, 1)
        lib.shim_fail_alloc(0)
        assert lib.gt_ens_run(e, 3) == 0 and lib.shim_bad() == 0
        assert lib.gt_ens_schedule(e, wide, 1) == 0 and lib.gt_ens_run(e, 3) == 0
        assert lib.gt_ens_destroy(e) == 0 and lib.shim_bad() == 0
        if rc == 0:
            break
    assert 20 < k < 99

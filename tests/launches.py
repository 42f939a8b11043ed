"""Records what the library's entry points launch, without a GPU.

The objects of libbpdq_hip.so are linked against the stand-in for the HIP runtime below:
a launch is written down (kernel, grid, block, dynamic LDS) instead of run, allocations are
host memory.  So a test sees the choice that the launchers really make for a shape.  The
kernels do not run and nothing reads their operands: any aligned address will do.
"""
import ctypes
import glob
import os
import re
import subprocess

from bpd_substrate_amd import _native, build

STUB = r"""
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>
struct Dim { uint32_t x, y, z; };
struct Launch { const char* name; uint32_t grid[3], block[3]; uint64_t lds; };
static std::map<const void*, std::string>& names() { static std::map<const void*, std::string> m; return m; }
static std::vector<Launch> log_;
static struct { Dim g, b; size_t lds; void* s; } cfg;
static char fat[64];
extern "C" {
void** __hipRegisterFatBinary(const void*) { return reinterpret_cast<void**>(fat); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    names()[f] = name;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim g, Dim b, size_t lds, void* s) { cfg = {g, b, lds, s}; return 0; }
int __hipPopCallConfiguration(Dim* g, Dim* b, size_t* lds, void** s) {
    *g = cfg.g; *b = cfg.b; *lds = cfg.lds; *s = cfg.s;
    return 0;
}
int hipLaunchKernel(const void* f, Dim g, Dim b, void**, size_t lds, void*) {
    log_.push_back({names()[f].c_str(), {g.x, g.y, g.z}, {b.x, b.y, b.z}, lds});
    return 0;
}
int hipFuncSetAttribute(const void*, int, int) { return 0; }
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return ""; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipDeviceSynchronize() { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamIsCapturing(void*, int* c) { *c = 0; return 0; }
int hipMalloc(void** p, size_t n) { *p = std::aligned_alloc(256, (n + 255) / 256 * 256); return *p == nullptr; }
int hipFree(void* p) { std::free(p); return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int) { std::memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { std::memcpy(d, s, n); return 0; }
int hipGetSymbolAddress(void** p, const void*) { *p = fat; return 0; }
const Launch* launches(int* n) { *n = (int)log_.size(); return log_.data(); }
void launches_clear() { log_.clear(); }
}
"""


class _Launch(ctypes.Structure):
    _fields_ = [("name", ctypes.c_char_p), ("grid", ctypes.c_uint32 * 3), ("block", ctypes.c_uint32 * 3),
                ("lds", ctypes.c_uint64)]


class Launch:
    """kernel: its name; args: its template arguments as ints (None where one is no number)."""

    def __init__(self, raw, demangled):
        m = re.match(r"(?:void )?(?:bpdq::)?(?:\(anonymous namespace\)::)?(\w+)(?:<(.*?)>)?\(", demangled)
        self.kernel = m.group(1)
        self.args = [_number(a) for a in (m.group(2) or "").split(",") if a.strip()]
        self.grid, self.block, self.lds = tuple(raw.grid), tuple(raw.block), raw.lds

    def __repr__(self):
        return f"{self.kernel}<{', '.join(map(str, self.args))}> {self.grid} x {self.block}, {self.lds} B"


def _number(a):
    a = a.strip()
    if a in ("true", "false"):
        return int(a == "true")
    return int(a) if re.fullmatch(r"-?\d+", a) else None


def _objects():
    objs = [os.path.join(build.OBJ, os.path.basename(s)[:-4] + ".o") for s in build.hip_sources()]
    newest = max(os.path.getmtime(f) for f in glob.glob(os.path.join(build.CSRC, "*")))
    if not all(os.path.exists(o) and os.path.getmtime(o) >= newest for o in objs):
        objs = build.compile_hip()
    return objs


class Recorder:
    def __init__(self, folder):
        src, so = os.path.join(folder, "hip_stub.cpp"), os.path.join(folder, "libbpdq_launches.so")
        with open(src, "w") as f:
            f.write(STUB)
        subprocess.run([build.CXX, "-std=c++17", "-O1", "-fPIC", "-shared", "-o", so, src, *_objects(), "-lm", "-lpthread"],
                       check=True)
        self.lib = _native._load(so, _native.HIP_SIGNATURES, "the launch recorder")
        self.lib.launches.restype = ctypes.POINTER(_Launch)
        self.names = {}

    def __call__(self, name, *args):
        """The launches of one call of entry point `name`."""
        self.lib.launches_clear()
        getattr(self.lib, name)(*args)
        err = self.lib.bpd_gpu_last_error()
        assert err == 0, (err, self.lib.bpd_gpu_last_error_message())
        n = ctypes.c_int()
        raw = self.lib.launches(ctypes.byref(n))
        return [Launch(raw[i], self._demangled(raw[i].name)) for i in range(n.value)]

    def _demangled(self, mangled):
        if mangled not in self.names:
            self.names[mangled] = subprocess.run(["c++filt", mangled.decode()], capture_output=True, text=True,
                                                 check=True).stdout.strip()
        return self.names[mangled]

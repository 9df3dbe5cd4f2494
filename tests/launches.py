"""Which kernels a call of the C interface launches, found on the host: the library runs in a process of its own against stand-ins for the HIP
runtime's entry points that write the launches down instead of making them."""
import ctypes
import json
import os
import subprocess
import sys
import tempfile

from flashdeberta_amd import _lib

STAND_INS = r"""
#include <cstddef>
#include <cstdlib>
#include <map>
#include <string>
struct Dim { unsigned x, y, z; };
static std::map<const void*, std::string>& names() { static std::map<const void*, std::string> m; return m; }
static std::string& made() { static std::string s; return s; }
static int fails = 0, cus = 256;
static Dim grid_, block_;
static size_t lds_;
static void* stream_;
static void* handle;
extern "C" {
void stand_in_set(int compute_units, int launches_that_fail) { cus = compute_units, fails = launches_that_fail, made().clear(); }
const char* stand_in_made() { return made().c_str(); }
void** __hipRegisterFatBinary(const void*) { return &handle; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { names()[f] = name; }
int __hipPushCallConfiguration(Dim g, Dim b, size_t lds, void* s) { grid_ = g, block_ = b, lds_ = lds, stream_ = s; return 0; }
int __hipPopCallConfiguration(Dim* g, Dim* b, size_t* lds, void** s) { *g = grid_, *b = block_, *lds = lds_, *s = stream_; return 0; }
static int last = 0;
int hipLaunchKernel(const void* f, Dim g, Dim b, void**, size_t, void*) {
  made() += names()[f] + " " + std::to_string(g.x) + " " + std::to_string(g.y) + " " + std::to_string(b.x) + "\n";
  return last = fails > 0 ? (--fails, 719) : 0;
}
int hipGetLastError() { const int e = last; last = 0; return e; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int* v, int, int) { *v = cus; return 0; }
int hipFuncSetAttribute(const void*, int, int) { return 0; }
int hipGetSymbolAddress(void** p, const void*) { *p = (void*)0x100000; return 0; }
const char* hipGetErrorString(int) { return "failed"; }
}
"""

CHILD = r"""
import ctypes, json, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)   # ahead of the HIP runtime in the search order
lib = ctypes.CDLL(sys.argv[2])
shim.stand_in_made.restype = ctypes.c_char_p
out = []
for name, args, cus, fails in json.load(sys.stdin):
    shim.stand_in_set(cus, fails)
    given = [ctypes.create_string_buffer(bytes.fromhex(a["bytes"])) if isinstance(a, dict) and "bytes" in a else ctypes.c_void_p(a["pointer"]) if isinstance(a, dict)
             else ctypes.c_int64(a) for a in args]
    f = getattr(lib, name)
    f.restype = ctypes.c_int
    out.append((f(*given), shim.stand_in_made().decode().split("\n")[:-1]))
json.dump(out, sys.stdout)
"""


class P(int):
    """An address."""


def launches(calls, cus=256, fails=0):
    """calls: (entry point, arguments: structures, P addresses, None or whole numbers).  Returns for each (its code, [(kernel, grid x, grid y,
    threads)]).  `cus`: compute units of the device; `fails`: so many launches of each call return an error (719)."""
    def pack(a):
        if isinstance(a, ctypes.Structure):
            return {"bytes": bytes(a).hex()}
        return {"pointer": None if a is None else int(a)} if a is None or isinstance(a, P) else int(a)

    with tempfile.TemporaryDirectory() as where:
        source, shim = os.path.join(where, "stand_ins.cpp"), os.path.join(where, "stand_ins.so")
        with open(source, "w") as f:
            f.write(STAND_INS)
        subprocess.run([os.environ.get("CXX", "g++"), "-shared", "-fPIC", "-O1", "-o", shim, source], check=True)
        todo = json.dumps([(name, [pack(a) for a in args], cus, fails) for name, args in calls])
        r = subprocess.run([sys.executable, "-c", CHILD, shim, _lib.LIB_PATH], input=todo, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    return [(rc, [(l.split()[0], *map(int, l.split()[1:])) for l in lines]) for rc, lines in json.loads(r.stdout)]

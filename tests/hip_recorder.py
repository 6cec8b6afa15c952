"""Host code without a GPU: the library's calls into the HIP runtime are answered by a small stand-in that notes every launch
(kernel, grid, block) and runs nothing, so that what an entry point launches for a geometry can be checked on the CPU."""
import json
import os
import subprocess
import sys
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cstdint>
#include <cstring>
#include <map>
#include <string>
struct Dim { uint32_t x, y, z; };
static std::map<const void *, std::string> &names() { static std::map<const void *, std::string> m; return m; }
static std::string noted;
static thread_local Dim grid_, block_;
static thread_local size_t lds_;
static thread_local void *stream_;
static int last_error;
static void note(const void *f, Dim g, Dim b) {
  auto it = names().find(f);
  noted += (it == names().end() ? std::string("?") : it->second) + " " + std::to_string(g.x) + " " + std::to_string(g.y) + " " +
           std::to_string(g.z) + " " + std::to_string(b.x * b.y * b.z) + "\n";
}
extern "C" {
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) { names()[host] = name; }
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim g, Dim b, size_t l, void *s) { grid_ = g, block_ = b, lds_ = l, stream_ = s; return 0; }
int __hipPopCallConfiguration(Dim *g, Dim *b, size_t *l, void **s) { *g = grid_, *b = block_, *l = lds_, *s = stream_; return 0; }
// (the runtime counts threads in 32 bits: a grid of more is refused)
static int launch(const void *f, Dim g, Dim b) {
  if (uint64_t(g.x) * b.x > 0xffffffffu || uint64_t(g.y) * b.y > 0xffffffffu || uint64_t(g.z) * b.z > 0xffffffffu || g.y > 65535 || g.z > 65535)
    return last_error = 9;
  note(f, g, b);
  return 0;
}
int hipLaunchKernel(const void *f, Dim g, Dim b, void **, size_t, void *) { return launch(f, g, b); }
int hipExtLaunchKernel(const void *f, Dim g, Dim b, void **, size_t, void *, void *, void *, int) { return launch(f, g, b); }
int hipGetLastError() { const int e = last_error; last_error = 0; return e; }
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int *v, int, int) { *v = 256; return 0; }
static std::string refused;   // kernels whose attributes are refused
void recorder_refuse(const char *part) { refused = part; }
int hipFuncSetAttribute(const void *f, int, int) { return !refused.empty() && names()[f].find(refused) != std::string::npos ? 1 : 0; }
const char *recorder_take() { static std::string out; out = noted; noted.clear(); return out.c_str(); }
}
"""

PREAMBLE = """
import ctypes as C, json, sys
sys.path[:0] = [%r, %r]
recorder = C.CDLL(%r, mode=C.RTLD_GLOBAL)
recorder.recorder_take.restype = C.c_char_p
from singa_amd import _lib
lib = _lib.lib()


def launched():
    '''[(mangled kernel name, (grid x, y, z), threads of a block)] since the last call'''
    out = []
    for l in recorder.recorder_take().decode().splitlines():
        f = l.rsplit(" ", 4)
        out.append((f[0], tuple(int(v) for v in f[1:4]), int(f[4])))
    return out


def kernels():
    '''the kernels' plain names, in order'''
    import re
    found = [(re.search(r"\\d(k_[a-z0-9_]+)", n), n) for n, _, _ in launched()]   # (a name ends at the I, E or P of the mangling)
    return [m.group(1) if m else n for m, n in found]


def conv(*dims):
    g = _lib.ConvGeom()
    assert lib.sgh_conv_geom_init(C.byref(g), *dims) == 0
    return g


SPACE = 1 << 40   # an address: nothing reads it
"""


def recorded(code):
    """What `code` hands to answer(...), run in a process of its own with the stand-in in front of the runtime."""
    with tempfile.TemporaryDirectory() as d:
        src, so = os.path.join(d, "recorder.cc"), os.path.join(d, "recorder.so")
        with open(src, "w") as f:
            f.write(SOURCE)
        subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", src, "-o", so])
        body = PREAMBLE % (ROOT, os.path.join(ROOT, "tests"), so) + "\ndef answer(v):\n    print('ANSWER ' + json.dumps(v), flush=True)\n\n" + code
        p = subprocess.run([sys.executable, "-c", body], stdout=subprocess.PIPE, stderr=subprocess.PIPE, timeout=120, cwd=ROOT)
        lines = [l for l in p.stdout.decode().splitlines() if l.startswith("ANSWER ")]
        assert p.returncode == 0 and lines, p.stderr.decode()[-3000:]
        return json.loads(lines[-1][7:])

"""Kernel launches of libmgp.so recorded instead of run, on the CPU: which kernel
serves a call, with what grid, block and dynamic LDS.

The recorder defines the launch functions of the HIP runtime and is loaded
before libmgp.so, whose launches then end in its list.  It lives in a process
of its own (record() starts one per set of calls), so nothing else sees it.
Array data pointers are never followed by the host code, so any non-zero value
stands for an array."""
import ctypes
import json
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))

RECORDER = r"""
#include <cstdint>
#include <cstdio>
#include <map>
#include <string>
struct dim3 { uint32_t x, y, z; };
static std::map<const void*, std::string> names;
static std::string list;
static dim3 cfg_grid, cfg_block;
static size_t cfg_lds;
static void* cfg_stream;
extern "C" {
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) { names[host] = name; }
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, void* stream) {
    cfg_grid = g, cfg_block = b, cfg_lds = lds, cfg_stream = stream;
    return 0;
}
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, void** stream) {
    *g = cfg_grid, *b = cfg_block, *lds = cfg_lds, *stream = cfg_stream;
    return 0;
}
int hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t lds, void*) {
    char s[64];
    std::snprintf(s, sizeof s, " %u %u %zu\n", g.x * g.y * g.z, b.x * b.y * b.z, lds);
    list += names[f] + s;
    return 0;
}
int hipGetLastError() { return 0; }
const char* recorded() { return list.c_str(); }
void forget() { list.clear(); }
}
"""


def build(folder):
    src, lib = os.path.join(folder, "recorder.cpp"), os.path.join(folder, "recorder.so")
    with open(src, "w") as f:
        f.write(RECORDER)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", src, "-o", lib], check=True)
    return lib


def record(lib, calls):
    """[(return code, [(kernel, workgroups, threads, LDS bytes)])] of `calls`,
    each a dict: name, arrays {argument name: (shape, halo, strides or None)}
    with the argument order in args (array names, numbers, or "faces" / "box"),
    bc, box, h and tuning keys."""
    r = subprocess.run([sys.executable, os.path.abspath(__file__), lib], input=json.dumps(calls), text=True,
                       capture_output=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return [(rc, [tuple(k) for k in kernels]) for rc, kernels in json.loads(r.stdout.splitlines()[-1])]


def _child(lib):
    rec = ctypes.CDLL(lib, mode=ctypes.RTLD_GLOBAL)
    rec.recorded.restype = ctypes.c_char_p
    sys.path.insert(0, os.path.join(os.path.dirname(HERE), "multigrid-poisson_amd"))
    import mgp

    L = mgp.lib()
    out = []
    for c in json.load(sys.stdin):
        arrays = {}
        for n, (name, (shape, halo, strides)) in enumerate(sorted(c["arrays"].items())):
            a = mgp.Array()
            a.data = (n + 1) << 44
            a.shape[:], a.halo[:] = shape, halo
            p = mgp.padded_shape(shape, halo)
            a.stride[:] = strides or [p[1] * p[2], p[2], 1]
            arrays[name] = a
        F = mgp.Faces()
        F.h = c["h"]
        for q in range(6):
            F.type[q] = mgp.NEUMANN if c["bc"][q] == "N" else mgp.DIRICHLET
            F.g[q] = (q + 32) << 44 if c["bc"][q] == "N" else None
        values = {"faces": ctypes.byref(F), "box": mgp.box(c["box"]), "stream": None}
        args = [ctypes.byref(arrays[v]) if v in arrays else values[v] if isinstance(v, str) else v for v in c["args"]]
        old = {}
        for key, v in c.get("keys", {}).items():
            cur = ctypes.c_int64()
            mgp.check(L.mgp_tuning_get(key.encode(), ctypes.byref(cur)))
            mgp.check(L.mgp_tuning_set(key.encode(), v))
            old[key] = cur.value
        rec.forget()
        rc = getattr(L, c["name"])(*args)
        kernels = []
        for line in rec.recorded().decode().splitlines():
            name, grid, block, lds = line.rsplit(" ", 3)
            kernels.append((name, int(grid), int(block), int(lds)))
        out.append((rc, kernels))
        for key, v in old.items():
            L.mgp_tuning_set(key.encode(), v)
    print(json.dumps(out))


if __name__ == "__main__":
    _child(sys.argv[1])

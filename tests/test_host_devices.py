"""A context serves its own device whatever device the calling thread has current, and leaves that device current: the
entry points run here against a stand-in for the HIP runtime with two devices, which records where they launch."""

import os
import re
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

STAND_IN = r"""
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
static int current = 0, switches = 0, seen[2] = {0, 0};
#define ON ++seen[current]
int hipGetDeviceCount(int* n) { *n = 2; return 0; }
int hipGetDevice(int* d) { *d = current; return 0; }
int hipSetDevice(int d) { current = d; ++switches; return 0; }
int fake_current(void) { return current; }
int fake_seen(int d) { return seen[d]; }
int fake_switches(void) { return switches; }
void fake_clear(void) { seen[0] = seen[1] = switches = 0; }
int hipGetDevicePropertiesR0600(void* p, int d) { memset(p, 0, 256); return 0; }
const char* hipGetErrorString(int e) { return "stand-in"; }
int hipGetLastError(void) { return 0; }
int hipMalloc(void** p, size_t n) { ON; *p = malloc(n); return *p ? 0 : 2; }
int hipFree(void* p) { ON; free(p); return 0; }
int hipMemset(void* p, int v, size_t n) { ON; return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) { ON; return 0; }
int hipDeviceSynchronize(void) { ON; return 0; }
int hipStreamCreate(void** s) { ON; *s = malloc(8); return 0; }
int hipStreamCreateWithFlags(void** s, unsigned f) { ON; *s = malloc(8); return 0; }
int hipStreamDestroy(void* s) { ON; free(s); return 0; }
int hipStreamSynchronize(void* s) { ON; return 0; }
int hipStreamIsCapturing(void* s, int* st) { *st = 0; return 0; }
int hipStreamBeginCapture(void* s, int m) { ON; return 0; }
int hipStreamEndCapture(void* s, void** g) { ON; *g = malloc(8); return 0; }
int hipGraphInstantiate(void** e, void* g, void** n, char* b, size_t z) { ON; *e = malloc(8); return 0; }
int hipGraphLaunch(void* e, void* s) { ON; return 0; }
int hipGraphDestroy(void* g) { ON; free(g); return 0; }
int hipGraphExecDestroy(void* e) { ON; free(e); return 0; }
int hipEventCreate(void** e) { ON; *e = malloc(8); return 0; }
int hipEventDestroy(void* e) { ON; free(e); return 0; }
int hipEventRecord(void* e, void* s) { ON; return 0; }
int hipEventSynchronize(void* e) { ON; return 0; }
int hipEventElapsedTime(float* t, void* a, void* b) { *t = 1.0f; return 0; }
int hipGetSymbolAddress(void** p, const void* s) { ON; *p = malloc(1 << 20); return 0; }
typedef struct { unsigned x, y, z; } dim3_;
int hipLaunchKernel(const void* f, dim3_ g, dim3_ b, void** a, size_t l, void* s) { ON; return 0; }
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t l, void* s) { return 0; }
int __hipPopCallConfiguration(dim3_* g, dim3_* b, size_t* l, void** s) { *l = 0; *s = 0; memset(g, 0, 12); memset(b, 0, 12); return 0; }
void** __hipRegisterFatBinary(const void* d) { static void* m; return &m; }
void __hipUnregisterFatBinary(void** m) {}
void __hipRegisterFunction(void) {}
void __hipRegisterVar(void) {}
"""

PROGRAM = r"""
import ctypes, sys
sys.path.insert(0, sys.argv[1])
fake = ctypes.CDLL(sys.argv[2], mode=ctypes.RTLD_GLOBAL)
from nofluidx3d_amd import _lib
L = ctypes.CDLL(_lib.LIB_PATH)
_lib._bind(L, _lib.SIGNATURES)
h = ctypes.c_void_p()
assert L.nfx_init(1, _lib.STREAM_DEFAULT, ctypes.byref(h)) == 0, L.nfx_last_error()

def inside(name, *args, refused=False):
    '''one call with device 0 current: its work is on device 1, and device 0 is current afterwards'''
    fake.hipSetDevice(0)
    fake.fake_clear()
    rc = getattr(L, name)(*args)
    assert (rc != 0) == refused, (name, rc, L.nfx_last_error())
    assert fake.fake_seen(0) == 0, f"{name} worked on the caller's device"
    assert fake.fake_switches() == 2, f"{name} changed the device {fake.fake_switches()} times"
    assert fake.fake_current() == 0, f"{name} left another device current"
    assert refused or fake.fake_seen(1) > 0, name

null = lambda t: t() if issubclass(t, ctypes._SimpleCData) else None
for name in sys.argv[3].split(","):  # every entry point, refused for its missing arguments
    inside(name, h, *[null(t) for t in _lib.SIGNATURES[name][1][1:]], refused=name != "nfx_stream_sync")

b = [ctypes.create_string_buffer(64) for _ in range(24)]
q = lambda i: ctypes.addressof(b[i])
inside("nfx_sphere_force", h, q(0), q(1), 4, 0.1, 1.0, 0.0)
inside("nfx_velocity_verlet", h, q(0), q(1), q(2), q(3), 4, 0)
inside("nfx_over_damped", h, q(0), q(1), 4, 0)
inside("nfx_mlp_mse", h, q(0), q(1), None, 32, 32, q(2), q(3), q(4))
p = _lib.Plan()
p.N, p.T = 4, 1
p.tetras, p.dminv, p.v0, p.ref, p.disp, p.vel, p.fold, p.force = (q(i) for i in range(8))
p.model, p.scatter = _lib.NFX_MR, _lib.SCATTER_TILED
p.tile_k, p.tile_max_nodes = 128, 4
p.tile_count, p.tile_nodes, p.tile_lend, p.tile_corners, p.tile_dst, p.node_off, p.partials = (q(i) for i in range(8, 15))
p.disp_b, p.vel_b, p.partials_b, p.tile_range = (q(i) for i in range(15, 19))
p.indenter, p.ind_k, p.ind_radius = _lib.INDENTER_SPHERE, 0.1, 1.0
inside("nfx_run_steps", h, ctypes.byref(p), 0, 300, q(19), 1)  # captures, replays and allocates
n = ctypes.c_int64()
assert L.nfx_graph_captures(h, ctypes.byref(n)) == 0 and n.value == 1
inside("nfx_destroy", h)
print("ok")
"""


def test_entry_points_work_on_the_contexts_device(tmp_path):
    src, lib = tmp_path / "hip.c", tmp_path / "libhip_stand_in.so"
    src.write_text(STAND_IN)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-w", "-o", str(lib), str(src)], check=True)
    header = open(os.path.join(ROOT, "include", "nfx.h")).read()
    names = re.findall(r"^int (nfx_\w+)\(nfx_ctx\* \w+[,)]", header, re.M)
    names = [n for n in names if n not in ("nfx_destroy", "nfx_graph_captures", "nfx_device_name")]
    assert len(names) > 30
    r = subprocess.run([sys.executable, "-c", PROGRAM, ROOT, str(lib), ",".join(names)], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr

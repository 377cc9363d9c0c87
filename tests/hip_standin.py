"""Runs host code of libmi_paged.so on the CPU against a stand-in HIP runtime that records launches.

``run(body)`` starts a fresh interpreter that loads the stand-in before the library (its symbols come first),
executes ``body`` with ``lib`` (the library, signatures declared), ``hip`` (the stand-in) and ``launches()``
(name, template arguments, grid and block of every launch since the last call) in scope, and returns what
``body`` leaves in ``result``.  No kernel runs: pointers handed to the library are never read.
"""

from __future__ import annotations

import json
import os
import subprocess
import sys
import tempfile
import textwrap
from pathlib import Path

REPO = Path(__file__).resolve().parents[1]

_SOURCE = r"""
#include <stddef.h>
#include <stdint.h>
#include <string.h>
typedef struct { uint32_t x, y, z; } dim3_t;
typedef struct { const char* name; dim3_t grid, block; size_t lds; int device; } launch_t;
enum { kMax = 4096 };
static struct { const void* fn; const char* name; } kernels[kMax];
static int n_kernels;
static launch_t log_[kMax];
static int n_log, device_, n_attr, cus_ = 256;
static int attr_device[kMax];
static const char* attr_name[kMax];
static dim3_t cfg_grid, cfg_block;
static size_t cfg_lds;
static void* cfg_stream;
static const char* name_of(const void* fn) {
  for (int i = 0; i < n_kernels; ++i) if (kernels[i].fn == fn) return kernels[i].name;
  return "?";
}
void** __hipRegisterFatBinary(const void* data) { (void)data; static void* handle; return &handle; }
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterFunction(void** m, const void* fn, char* dev, const char* name, unsigned limit, void* tid, void* bid,
                           void* bd, void* gd, int* ws) {
  (void)m; (void)dev; (void)limit; (void)tid; (void)bid; (void)bd; (void)gd; (void)ws;
  if (n_kernels < kMax) { kernels[n_kernels].fn = fn; kernels[n_kernels++].name = name; }
}
void __hipRegisterVar(void** m, void* v, char* h, char* d, int e, size_t s, int c, int g) {
  (void)m; (void)v; (void)h; (void)d; (void)e; (void)s; (void)c; (void)g;
}
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t lds, void* s) {
  cfg_grid = g; cfg_block = b; cfg_lds = lds; cfg_stream = s; return 0;
}
int __hipPopCallConfiguration(dim3_t* g, dim3_t* b, size_t* lds, void** s) {
  *g = cfg_grid; *b = cfg_block; *lds = cfg_lds; *s = cfg_stream; return 0;
}
int hipLaunchKernel(const void* fn, dim3_t g, dim3_t b, void** args, size_t lds, void* s) {
  (void)args; (void)s;
  if (n_log < kMax) { launch_t l = {name_of(fn), g, b, lds, device_}; log_[n_log++] = l; }
  return 0;
}
int hipFuncSetAttribute(const void* fn, int attr, int value) {
  (void)attr; (void)value;
  if (n_attr < kMax) { attr_name[n_attr] = name_of(fn); attr_device[n_attr++] = device_; }
  return 0;
}
int hipGetDevice(int* d) { *d = device_; return 0; }
int hipDeviceGetAttribute(int* v, int attr, int dev) { (void)attr; (void)dev; *v = cus_; return 0; }
int hipGetLastError(void) { return 0; }
const char* hipGetErrorString(int e) { (void)e; return "stand-in"; }
int hipGetSymbolAddress(void** p, const void* s) { (void)s; static char scratch[256]; *p = scratch; return 0; }
void standin_set_device(int d) { device_ = d; }
void standin_reset(void) { n_log = n_attr = 0; }
int standin_launches(void) { return n_log; }
const launch_t* standin_launch(int i) { return &log_[i]; }
int standin_attrs(void) { return n_attr; }
const char* standin_attr_name(int i) { return attr_name[i]; }
int standin_attr_device(int i) { return attr_device[i]; }
"""

_PRELUDE = r"""
import ctypes, json, re, sys, types
sys.path.insert(0, {repo!r})
hip = ctypes.CDLL({standin!r}, mode=ctypes.RTLD_GLOBAL)
sys.modules["torch"] = types.ModuleType("torch")  # the binding only orders its import
from mini_infra_qwen3_amd import _native
class Launch(ctypes.Structure):
    _fields_ = [("name", ctypes.c_char_p), ("grid", ctypes.c_uint32 * 3), ("block", ctypes.c_uint32 * 3),
                ("lds", ctypes.c_size_t), ("device", ctypes.c_int)]
hip.standin_launch.restype = ctypes.POINTER(Launch)
hip.standin_attr_name.restype = ctypes.c_char_p
lib = ctypes.CDLL(str(_native.LIBRARY_PATH))
for _name, (_res, _args) in _native.SIGNATURES.items():
    getattr(lib, _name).restype, getattr(lib, _name).argtypes = _res, _args
def kernel(mangled):
    m = re.search(r"\d+([a-z_]+_kernel)(?:I(.*?)EEv|E)", mangled)
    args = [int(x) for x in re.findall(r"L[ib](\d+)E", m.group(2) + "E")] if m and m.group(2) else []
    return m.group(1) if m else mangled, args
def launches():
    out = []
    for i in range(hip.standin_launches()):
        l = hip.standin_launch(i).contents
        name, args = kernel(l.name.decode())
        out.append(dict(kernel=name, args=args, grid=list(l.grid), block=l.block[0], lds=l.lds, device=l.device,
                        mangled=l.name.decode()))
    hip.standin_reset()
    return out
result = None
"""


def run(body: str):
    from mini_infra_qwen3_amd import _native, build

    if not _native.LIBRARY_PATH.exists():
        build.build(verbose=False)
    with tempfile.TemporaryDirectory() as tmp:
        source, standin = Path(tmp, "standin.c"), Path(tmp, "libstandin.so")
        source.write_text(_SOURCE)
        subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(standin), str(source)], check=True)
        script = _PRELUDE.format(repo=str(REPO), standin=str(standin)) + textwrap.dedent(body) + \
            "\nprint('RESULT ' + json.dumps(result), flush=True)\n"
        env = {k: v for k, v in os.environ.items() if k != "MI_DECODE_PATH"}
        proc = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True, timeout=120, env=env)
    lines = [line for line in proc.stdout.splitlines() if line.startswith("RESULT ")]
    assert proc.returncode == 0 and lines, proc.stdout + proc.stderr
    return json.loads(lines[-1][len("RESULT "):])

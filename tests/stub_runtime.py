"""Runs a script in a process whose libamps.so is bound to tests/hip_stub.c in
place of the HIP runtime: kernels are logged, not run.  The script finds
`amps` (the package), `stub` (live(), peak(), limit(bytes), clear() and
log(): the kernels launched, "graph" for a replayed graph, "copy", "memset",
"free" and "host" (a host function), a leading + while a graph is captured) and `out`, a dict that comes back."""
import json
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

GRAPH = ["hipStreamBeginCapture", "hipStreamEndCapture", "hipGraphInstantiate", "hipGraphDestroy",
         "hipGraphExecDestroy", "hipGraphLaunch"]

PRELUDE = """
import ctypes, json, sys
sys.path.insert(0, {root!r})
class Stub:
    def __init__(self):
        self.h = ctypes.CDLL({lib!r}, mode=ctypes.RTLD_GLOBAL)
        self.h.stub_log.restype = ctypes.c_char_p
        self.h.stub_live.restype = self.h.stub_peak.restype = ctypes.c_size_t
        self.h.stub_limit.argtypes = [ctypes.c_size_t]
    def log(self): return self.h.stub_log().decode().split()
    def clear(self): self.h.stub_clear()
    def live(self): return self.h.stub_live()
    def peak(self): return self.h.stub_peak()
    def limit(self, n): self.h.stub_limit(n)
stub = Stub()
import w3914777_amd as amps
out = {{}}
"""


def build(tmp):
    lib, ver = os.path.join(tmp, "libhipstub.so"), os.path.join(tmp, "hip.map")
    with open(ver, "w") as f:
        f.write("hip_4.2 { global: *; };\nhip_4.3 { global: " + " ".join(g + ";" for g in GRAPH) + " } hip_4.2;\n"
                "hip_5.3 { global: hipLaunchHostFunc; } hip_4.3;\n")
    subprocess.run(["gcc", "-O1", "-Wall", "-shared", "-fPIC", os.path.join(HERE, "hip_stub.c"), "-o", lib,
                    "-Wl,-soname,libamdhip64.so.7", "-Wl,--version-script," + ver], check=True)
    return lib


def run(lib, script):
    code = PRELUDE.format(root=ROOT, lib=lib) + script + "\nprint('OUT ' + json.dumps(out))\n"
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    m = re.search(r"^OUT (.*)$", r.stdout, re.M)
    assert r.returncode == 0 and m, r.stdout + r.stderr
    return json.loads(m.group(1))

"""What libr9vx launches for a call, recorded on the CPU: the library runs in a
child process on tests/fixtures/record_amdhip64.c instead of the HIP runtime.
No device is touched and no argument is dereferenced."""
from __future__ import annotations

import json
import os
import pathlib
import re
import subprocess
import sys

ROOT = pathlib.Path(__file__).resolve().parents[1]
LIB = ROOT / "r9v_amd" / "libr9vx.so"
SOURCE = ROOT / "tests" / "fixtures" / "record_amdhip64.c"
SYMBOLS = re.findall(r"^(?!static)\w[\w* ]*?(\w+)\([^;{)]*\) \{", SOURCE.read_text(), re.M)

CHILD = r'''
import ctypes, json, sys
from r9v_amd import ffi
L = ffi.load()
hip = ctypes.CDLL("libamdhip64.so.7")
FAKE = ctypes.c_void_p(1 << 20)  # 256-byte aligned; nothing reads it

def launches():
    out, i = [], 0
    name, g, b = ctypes.c_char_p(), (ctypes.c_uint32 * 3)(), (ctypes.c_uint32 * 3)()
    while hip.recorded(i, ctypes.byref(name), g, b):
        out.append([name.value.decode(), list(g), list(b)])
        i += 1
    hip.record_clear()
    return out

def matmul(scheme, m, n, k, m_bucket=None, x_f32=False, bf16_out=False, epilogue=0, tiles=None):
    st = ffi.matmul_static(n=n, k=k, w_scheme=scheme, in_dtype=ffi.F32 if x_f32 else ffi.BF16,
                           out_dtype=ffi.BF16 if bf16_out else ffi.F32, m_bucket=m_bucket or m, epilogue=epilogue)
    split = scheme in ffi.SPLIT_SCHEMES
    args = ffi.MatmulArgs(FAKE, FAKE if split else None, None, FAKE, None, FAKE if epilogue == 1 else None,
                          FAKE if epilogue == 2 else None, FAKE, FAKE, m, 0)
    if tiles:
        return L.r9vx_probe_matmul_tiles_launch(ctypes.byref(st), ctypes.byref(args), *tiles, None)
    return L.r9vx_matmul_launch(ctypes.byref(st), ctypes.byref(args), None)

def route(t, e, k, scoring=0):
    st = ffi.route_static(e=e, k=k, t_bucket=t, scoring=scoring)
    args = ffi.MoeRouteArgs(FAKE, None, FAKE, FAKE, t, 0)
    return L.r9vx_moe_route_launch_ex(ctypes.byref(st), ctypes.byref(args), FAKE, None)

out = []
for f, kw in json.loads(sys.argv[1]):
    rc = globals()[f](**kw)
    out.append([rc, L.r9vx_last_error().decode() if rc else "", launches()])
print(json.dumps(out))
'''


def build(directory):
    """The stand-in runtime, built into `directory`."""
    version = directory / "hip.map"
    version.write_text("hip_4.2 {\n  global:\n" + "".join(f"    {s};\n" for s in SYMBOLS) + "  local: *;\n};\n")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-Wl,-soname,libamdhip64.so.7",
                    f"-Wl,--version-script={version}", "-o", str(directory / "libamdhip64.so.7"), str(SOURCE)], check=True)
    return directory


def record(directory, calls):
    """[(return code, error text, [(kernel, grid, block), ...])] of `calls`, each
    (function of the child, keyword arguments), on the runtime in `directory`."""
    env = dict(os.environ, LD_LIBRARY_PATH=str(directory), PYTHONPATH=str(ROOT))
    r = subprocess.run([sys.executable, "-c", CHILD, json.dumps(calls)], env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    out = json.loads(r.stdout.strip().splitlines()[-1])
    return [(rc, msg, [(kernel_name(n), g, b) for n, g, b in ls]) for rc, msg, ls in out]


def kernel_name(mangled):
    """`kernel<1, 2>` of a mangled kernel name (c++filt, without the argument list)."""
    text = subprocess.run(["c++filt", mangled], capture_output=True, text=True, check=True).stdout.strip()
    text = re.sub(r"^void ", "", text).replace("(anonymous namespace)::", "")
    return re.sub(r"\(\w[^()]*\)$|\(\)$", "", text)

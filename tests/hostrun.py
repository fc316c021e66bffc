"""Runs a piece of Python against the library with the recording HIP runtime of host_hip/host_hip.cpp, in a process
of its own (a GPU is neither needed nor touched)."""
import os
import subprocess
import sys
import textwrap

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes, os, sys
sys.modules["torch"] = None  # the library's HIP symbols are to resolve to the recording runtime
sys.path[:0] = [%(root)r]
H = ctypes.CDLL(%(hip)r, mode=ctypes.RTLD_GLOBAL)
H.host_hip_log.restype = ctypes.c_char_p
from inductioneq_amd import _capi
from inductioneq_amd.schedules import rk_schedule
from inductioneq_amd.settings import ProgramConfig
lib = _capi.load()
P = ctypes.c_void_p


def build(**kw):
    cfg = ProgramConfig(**{"w_size": 64, **kw})
    h, mods = P(), cfg.modules()
    arr = (ctypes.c_char_p * len(mods))(*[m.encode() for m in mods])
    assert lib.ieq_program_build(ctypes.byref(h), cfg.settings_string().encode(), arr, len(mods)) == 0, lib.ieq_last_error(None)
    return h


def run(h, names, args, g):
    names = [names] if isinstance(names, str) else names
    cn = (ctypes.c_char_p * len(names))(*[n.encode() for n in names])
    return lib.ieq_run(h, cn, len(names), (ctypes.c_uint32 * 3)(*g), (ctypes.c_uint32 * 3)(64, 1, 1),
                       (P * len(args))(*args), len(args), None)


def log(*what):  # recorded lines that begin with one of `what`, split
    return [l.split() for l in H.host_hip_log().decode().splitlines() if not what or l.split()[0] in what]


def fail(fn, nth=1, code=719):
    H.host_hip_fail(fn.encode(), nth, code)


def far(n):  # n distinct addresses that nothing reads
    return [(k + 1) << 42 for k in range(n)]
"""


def build_hip(folder):
    from inductioneq_amd import _capi, build

    if not os.path.exists(_capi.LIB_PATH):
        build.build(verbose=False)
    so = os.path.join(str(folder), "host_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "host_hip", "host_hip.cpp"), "-o", so], check=True)
    return so


def hostrun(so, body, **env):
    src = PRELUDE % {"root": ROOT, "hip": so} + textwrap.dedent(body)
    e = {k: v for k, v in os.environ.items() if not k.startswith("IEQ_")}
    r = subprocess.run([sys.executable, "-c", src], capture_output=True, text=True, timeout=300, env={**e, **env})
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    return r.stdout

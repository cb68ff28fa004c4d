"""Runs host code of the native library without a GPU, on the HIP runtime of
fake_hip.cpp: run(script) starts a Python process in which that runtime is
loaded first, and returns what the script printed.  In the script, `fake` is
the runtime's control interface and log() its log, one list of words a call."""
import os
import subprocess
import sys

from conftest import ROOT

_PRELUDE = """
import ctypes, sys
sys.path[:0] = [%(root)r, %(tests)r]
fake = ctypes.CDLL(%(so)r, ctypes.RTLD_GLOBAL)
fake.fake_log.restype = ctypes.c_size_t
fake.fake_log.argtypes = [ctypes.c_char_p, ctypes.c_size_t]
fake.fake_live.restype = ctypes.c_uint64
fake.fake_refuse.argtypes = [ctypes.c_uint64, ctypes.c_uint64]
NEVER = 2 ** 64 - 1
WAIT = ctypes.CFUNCTYPE(None)
fake.fake_wait.argtypes = [ctypes.c_uint, ctypes.c_void_p]

def log():
    b = ctypes.create_string_buffer(fake.fake_log(None, 0) + 4096)
    fake.fake_log(b, len(b))
    return [l.split() for l in b.value.decode().splitlines()]

def launches(entries, name):
    return [e for e in entries if e[1] == "launch" and name in e[5]]

import numpy as np
from analisi_amd import capi
"""


def _library(folder):
    so = os.path.join(folder, "libfakehip.so")
    if not os.path.exists(so):
        subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", so], check=True)
    return so


def run(script, tmp_path_factory, timeout=120):
    so = _library(str(tmp_path_factory.getbasetemp()))
    text = _PRELUDE % dict(root=ROOT, tests=os.path.join(ROOT, "tests"), so=so) + script
    p = subprocess.run([sys.executable, "-c", text], capture_output=True, text=True, timeout=timeout, cwd=ROOT)
    assert p.returncode == 0, p.stdout + p.stderr
    return p.stdout

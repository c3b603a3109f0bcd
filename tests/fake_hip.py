"""Runs a piece of test code against the HIP library on a fake HIP runtime
(fake_hip.cpp), in a process of its own: the fake is loaded under the
runtime's name before the library is."""
import os
import subprocess
import sys
import textwrap

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_SONAME = "libamdhip64.so.7"

_PRELUDE = """
import ctypes as C, sys
sys.path.insert(0, {root!r})
fake = C.CDLL({lib!r}, mode=C.RTLD_GLOBAL)
fake.fake_count.restype = C.c_longlong
fake.fake_free_bytes.argtypes = [C.c_size_t]
fake.fake_fail.argtypes = [C.c_char_p, C.c_longlong]
fake.fake_launches.restype = C.c_longlong
launches = lambda part: fake.fake_launches(part.encode())
count = lambda name: fake.fake_count(name.encode())
import numpy as np
import cudasphnew_amd as S
from cudasphnew_amd import Field
"""


def build(folder) -> str:
    lib = os.path.join(str(folder), _SONAME)
    src = os.path.join(ROOT, "tests", "fake_hip.cpp")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", f"-Wl,-soname,{_SONAME}", src, "-o", lib],
                   check=True, capture_output=True)
    return lib


def run(lib: str, code: str) -> None:
    p = subprocess.run([sys.executable, "-c", _PRELUDE.format(root=ROOT, lib=lib) + textwrap.dedent(code)],
                       capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout + p.stderr

"""Runs a piece of Python against libawk_hip.so on a HIP runtime that only keeps books
(cxx/fake_hip.cpp), in a process of its own: no GPU, no kernel runs."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_HEAD = """
import ctypes, importlib.util
fake = ctypes.CDLL({fake!r}, mode=ctypes.RTLD_GLOBAL)
fake.fake_log.restype = ctypes.c_char_p
fake.fake_budget.argtypes = [ctypes.c_ulonglong]
fake.fake_used.restype = ctypes.c_ulonglong
spec = importlib.util.spec_from_file_location("_lib", {lib!r})
_lib = importlib.util.module_from_spec(spec)
spec.loader.exec_module(_lib)
lib = _lib.load()
P = ctypes.c_void_p

def log(kind=None):
    rows = [r.split(" ") for r in fake.fake_log().decode().splitlines()]
    return [r for r in rows if kind is None or r[0] == kind]

"""


def build(tmp):
    out = os.path.join(str(tmp), "fake_hip.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           os.path.join(ROOT, "tests", "cxx", "fake_hip.cpp"), "-o", out])
    return out


def run(fake, body):
    """The body's printed output; its assertions raise here."""
    head = _HEAD.format(fake=fake, lib=os.path.join(ROOT, "atlaswerks_amd", "_lib.py"))
    r = subprocess.run([sys.executable, "-c", head + body], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout

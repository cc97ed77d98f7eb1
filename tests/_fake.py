"""Runs a piece of Python against the engine's library on the stand-in for the HIP
runtime (cpp/fake_hip.cpp): host code on the CPU, no kernels.  In a process of its
own, since the stand-in has to be loaded before the engine."""
import subprocess
import sys
from pathlib import Path

TESTS = Path(__file__).resolve().parent
LIB = TESTS / "_build" / "libfake_hip.so"

PRELUDE = f"""
import ctypes as C, sys
fake = C.CDLL({str(LIB)!r}, mode=C.RTLD_GLOBAL)
fake.fake_log.restype = C.c_char_p
fake.fake_used.restype = C.c_size_t
fake.fake_fail.argtypes = [C.c_char_p, C.c_int]
fake.fake_limit.argtypes = [C.c_size_t]
sys.path.insert(0, {str(TESTS)!r})
from conftest import load_engine
vg = load_engine()
ctx = vg.Context(0)

def log():
    return fake.fake_log().decode().splitlines()

def launches():
    return [l.split()[1] for l in log() if l.startswith("launch")]

def sc(n, spin=vg.ISING, proposal=vg.FLIP, kind=vg.SC, seed=1):
    n = n if isinstance(n, tuple) else (n, n, n)
    return vg.chain(vg.lattice(kind, *n), spin, proposal, vg.hamiltonian(exchange=1.0), seed)
"""


def run(code: str) -> str:
    """Runs PRELUDE and code; what it printed.  Fails the test if it fails."""
    if not LIB.exists():
        subprocess.run(["make", "-s", "-C", str(TESTS / "cpp"), str(LIB)], check=True)
    r = subprocess.run([sys.executable, "-c", PRELUDE + code], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout

"""The library's host code on a HIP runtime that runs no kernels (native/fake_hip.cpp).

A scenario is a piece of Python run in a process of its own, with `rt` (the
runtime module on the fake), `lib` (its C library), `fake` (the fake's
controls), `np`, `C` and the helpers below in its names; what it assigns to
`result` comes back through JSON.
"""
from __future__ import annotations

import json
import shutil
import subprocess
import sys
import textwrap
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

PRELUDE = '''
import ctypes as C, json, sys, threading
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
fake.fake_log.restype = C.c_size_t
fake.fake_log.argtypes = [C.c_char_p, C.c_size_t]
fake.fake_set_malloc_limit.argtypes = [C.c_size_t]
import numpy as np
from leaf_amd import runtime as rt
lib = rt.library()

def log():
    """[(what, thread, ...)] since the last call: launches as ("launch", thread, kernel, stream, x, y, z)."""
    buffer = C.create_string_buffer(1 << 22)
    n = fake.fake_log(buffer, len(buffer))
    fake.fake_reset()
    return [line.split() for line in buffer.raw[:n].decode().splitlines()]

def kernels():
    """The kernels launched since the last call: their mangled names."""
    return [e[2] for e in log() if e[0] == "launch"]

buffer = rt.DeviceArray((1 << 20,), np.float32)     # an address: no kernel runs

def attention(tokens, position, heads=14, kv=2, dim=64, window=0, stream=None, q=None, out=None):
    return lib.lh_attention(q or buffer.ptr, buffer.ptr, buffer.ptr, position + tokens, heads, kv, dim, tokens,
                            position, window, out or buffer.ptr, stream)

def weight(bits, rows, cols, group=0):
    return rt.Weight(buffer.ptr, buffer.ptr if bits <= 8 else None, None, rows, cols, bits,
                     (group or cols) if bits <= 8 else 0)
'''


def run(scenario: str, library: Path, *args: str):
    code = PRELUDE + textwrap.dedent(scenario) + "\nprint('RESULT ' + json.dumps(result))\n"
    done = subprocess.run([sys.executable, "-c", code, str(library), *args], cwd=ROOT, capture_output=True, text=True,
                          timeout=120)
    assert done.returncode == 0, done.stderr
    return json.loads(done.stdout.rsplit("RESULT ", 1)[1])


@pytest.fixture(scope="session")
def fake_hip(tmp_path_factory):
    """run(scenario): what the scenario's `result` was."""
    if not shutil.which("g++"):
        pytest.skip("g++ is not installed")
    from leaf_amd import runtime
    if not runtime.LIBRARY.exists():
        pytest.skip("libleafhip.so is not built")
    library = tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", str(ROOT / "tests" / "native" / "fake_hip.cpp"),
                    "-o", str(library), "-lpthread"], check=True)
    return lambda scenario, *args: run(scenario, library, *args)

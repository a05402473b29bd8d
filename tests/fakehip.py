"""Runs a piece of Python against libmcm.so on the stand-in HIP runtime of
tests/fake_hip (no kernel runs, no GPU is needed), in a process of its own."""
from __future__ import annotations

import json
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
FAKE = os.path.join(HERE, "_build", "libfake_hip.so")
LIBMCM = os.path.join(os.path.dirname(HERE), "mcmatlab_amd", "libmcm.so")
needed = pytest.mark.skipif(not (os.path.exists(FAKE) and os.path.exists(LIBMCM)), reason="libmcm.so or the test harnesses not built")

PRELUDE = """
import ctypes as C, json, sys
sys.path[:0] = [{root!r}, {here!r}]
fake = C.CDLL({fake!r}, mode=C.RTLD_GLOBAL)
fake.fake_log.restype = C.c_char_p
fake.fake_peak.restype = C.c_size_t
fake.fake_set_limit.argtypes = [C.c_size_t]
import numpy as np
from mcmatlab_amd import _lib, abi, api
def log(clear=1):
    return fake.fake_log(clear).decode().split("\\n")[:-1]
def launches(lines):
    return [l.split()[1] for l in lines if l.startswith("launch ")]
def result(**kw):
    print("RESULT " + json.dumps(kw))
"""


def run(script):
    """The keyword arguments that the script gives to result()."""
    code = PRELUDE.format(root=os.path.dirname(HERE), here=HERE, fake=FAKE) + textwrap.dedent(script)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, f"exit {r.returncode}\n{r.stdout}\n{r.stderr}"
    return json.loads([ln for ln in r.stdout.splitlines() if ln.startswith("RESULT ")][-1][7:])

"""Runs a piece of Python in a process of its own with the library's device functions replaced by ones that note their calls
(cxx/recorded_calls.cpp): the order in which the host layer calls them, and what it does while it waits, without a GPU."""
import functools
import json
import os
import re
import subprocess
import sys
import tempfile

TESTS = os.path.dirname(os.path.abspath(__file__))
INCLUDE = os.path.join(os.path.dirname(TESTS), "include")

PRELUDE = """
import ctypes as C, json, os, sys, time
sys.path.insert(0, {tests!r})
stand_in = C.CDLL({library!r}, os.RTLD_GLOBAL | os.RTLD_NOW)
stand_in.recorded_name.restype = C.c_char_p
stand_in.recorded_stream.restype = C.c_void_p
stand_in.recorded_weights.argtypes, stand_in.recorded_weights.restype = [C.c_void_p], C.c_size_t
import lcu
P = lcu.package()
def calls():
    out = [(stand_in.recorded_name(i).decode(), stand_in.recorded_stream(i)) for i in range(stand_in.recorded_count())]
    stand_in.recorded_clear()
    return out
def tiny_model():
    return P.Model(dim=256, multiple_of=128, n_heads=2, n_layers=2, n_vocab=512, seed=1, weight_std=0.05, q_type=0, qblock=128)
"""


@functools.lru_cache(None)
def _library():
    folder = tempfile.mkdtemp()
    source = open(os.path.join(TESTS, "cxx", "recorded_calls.cpp")).read()
    header = re.sub(r"/\*.*?\*/", "", open(os.path.join(INCLUDE, "llama_cu_hip.h")).read(), flags=re.S)
    with open(os.path.join(folder, "other_calls.inc"), "w") as f:
        for result, name, arguments in re.findall(r"^(int|size_t) (lcu_\w+)\(([^)]*)\);", header, flags=re.M):
            if not re.search(r"\b%s\(" % name, source):
                stream = "stream" if re.search(r"void\* stream\b", arguments) else "nullptr"
                f.write('%s %s(%s) { return note("%s", %s); }\n' % (result, name, arguments, name, stream))
    path = os.path.join(folder, "recorded_calls.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-shared", "-fPIC", "-I", INCLUDE, "-I", folder,
                    os.path.join(TESTS, "cxx", "recorded_calls.cpp"), "-o", path], check=True)
    return path


def run(script):
    """What `script` leaves in `result`."""
    text = PRELUDE.format(tests=TESTS, library=_library()) + script + "\nprint(json.dumps(result))\n"
    done = subprocess.run([sys.executable, "-c", text], capture_output=True, text=True, timeout=120)
    assert done.returncode == 0, done.stderr
    return json.loads(done.stdout.splitlines()[-1])

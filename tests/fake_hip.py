"""The host code of a library on tests/cpp/fake_hip.cpp: a child process that runs no kernel and says what it would have launched."""
import json
import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent

PROLOGUE = """
import ctypes, json, sys
sys.path.insert(0, {root!r})
fake = ctypes.CDLL({library!r}, ctypes.RTLD_GLOBAL)
fake.fake_hip_log.restype = ctypes.c_char_p
def log(clear=True):
    lines = [l.split() for l in fake.fake_hip_log().decode().splitlines()]
    if clear:
        fake.fake_hip_clear()
    return lines
def answer(value):
    print("ANSWER " + json.dumps(value))
"""


def run(tmp_path, body):
    """What the Python text `body` hands to answer(); log() are the calls since it was last asked, as lists of words:
    launch or captured (kernel, grid, threads, dynamic LDS), lds (kernel, bytes), begin, end, instantiate, destroy, replay."""
    library = tmp_path / "libfake_hip.so"
    if not library.exists():
        subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(ROOT / "tests" / "cpp" / "fake_hip.cpp"), "-o", str(library)], check=True)
    proc = subprocess.run([sys.executable, "-c", PROLOGUE.format(root=str(ROOT), library=str(library)) + body], capture_output=True, text=True, timeout=120)
    assert proc.returncode == 0, proc.stderr[-3000:]
    return json.loads(next(l for l in proc.stdout.splitlines() if l.startswith("ANSWER "))[7:])

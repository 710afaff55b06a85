"""Runs a script against the library on the stand-in runtime of host_runtime.c,
in a process of its own (a process has one runtime).

The script sees `pkg` (the package), `P` (its parameter module), `rt` (the
stand-in: rt.mallocs, rt.live, rt.fail_at, rt.bad, rt.device as properties,
rt.launches() the recorded launches) and prints one line of JSON."""
import json
import os
import pathlib
import subprocess
import sys
import tempfile

from conftest import ROOT

HERE = pathlib.Path(__file__).resolve().parent

PRELUDE = """
import ctypes, json, subprocess, sys
sys.modules["torch"] = None  # its own runtime stays out of this process
sys.path.insert(0, {here!r})
from conftest import load_pkg, load_params
_lib = ctypes.CDLL({so!r}, ctypes.RTLD_GLOBAL)
_lib.host_log.restype = ctypes.c_char_p


class Runtime:
    def __getattr__(self, name):
        return ctypes.c_int.in_dll(_lib, "host_" + name).value

    def __setattr__(self, name, value):
        ctypes.c_int.in_dll(_lib, "host_" + name).value = value

    def log(self):
        return _lib.host_log().decode().splitlines()

    def clear(self):
        _lib.host_log_clear()

    def launches(self):
        out = []
        for line in self.log():
            w = line.split()
            if w[0] == "launch":
                out.append(dict(name=w[1], grid=tuple(map(int, w[3:6])), block=int(w[7]), lds=int(w[9]),
                                stream=w[11], device=int(w[13])))
        return out


rt = Runtime()
pkg, P = load_pkg(), load_params()
"""


def host_run(script):
    with tempfile.TemporaryDirectory() as d:
        so = pathlib.Path(d) / "host_runtime.so"
        subprocess.run(["gcc", "-O1", "-shared", "-fPIC", str(HERE / "host_runtime.c"), "-o", str(so)], check=True)
        env = dict(os.environ, PYTHONDONTWRITEBYTECODE="1")
        r = subprocess.run([sys.executable, "-c", PRELUDE.format(here=str(HERE), so=str(so)) + script],
                           cwd=ROOT, env=env, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return json.loads(r.stdout.strip().splitlines()[-1])

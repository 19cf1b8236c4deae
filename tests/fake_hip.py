"""Runs host code of the libraries in a child process on tests/fake_hip.c instead of the
HIP runtime, and works out from its log what the host has waited for."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes, sys
import numpy as np
sim = ctypes.CDLL({lib!r})
sim.hip_log.restype = ctypes.c_char_p
sim.hip_capture.argtypes = [ctypes.c_void_p, ctypes.c_int]
from fake_hip import Order
from gtt import capi
from helpers import angles_full, geom
L = capi.load()
S1, S2, S3 = 0x1000, 0x2000, 0x3000          # streams are names


def log():
    return sim.hip_log().decode().splitlines()


def count(what):
    return sum(l.split()[0] == what for l in log())


def limit(nbytes):
    ctypes.c_size_t.in_dll(sim, "hip_limit").value = nbytes


def context(angles=None, filt=None):
    h = ctypes.c_void_p()
    assert L.cbct_ctx_create(0, ctypes.byref(h)) == 0
    if angles is not None:
        views(h, angles)
    if filt:
        set_filter(h, filt)
    return h


def views(h, angles, offsets=None):
    a = np.ascontiguousarray(angles, np.float32)
    o = None if offsets is None else np.ascontiguousarray(offsets, np.float32)
    return L.cbct_views_set(h, a.ctypes.data, None if o is None else o.ctypes.data, len(a))


def set_filter(h, nu):
    F = np.arange(nu + 1, dtype=np.float32)
    return L.cbct_filter_set(h, nu, F.ctypes.data)


A = 0x10000                                  # arrays that kernels would use are names, too


def fp(h, g, n, stream, view0=0):
    return L.cbct_fp(h, ctypes.byref(g), view0, n, A, 0, A, 1.5, 0, stream)


def fp_noalloc(h, g, n, stream):
    return L.cbct_fp_noalloc(h, ctypes.byref(g), 0, n, A, 0, A, 1.5, 0, stream)


def bp(h, g, n, stream):
    return L.cbct_bp(h, ctypes.byref(g), 0, n, A, 0, A, 0, 0, stream)


def prefilter(h, g, n, stream):
    return L.cbct_fdk_prefilter(h, ctypes.byref(g), 0, n, A, A, 0, 0, stream)
"""


class Order:
    """For every line of a log, which launches the host has waited for."""

    def __init__(self, log):
        streams, events, host = {}, {}, set()
        self.launches, self.unwaited = [], []   # per copy to the device: launches not waited for
        for i, line in enumerate(log):
            w = line.split()
            if w[0] == "launch":
                streams.setdefault(w[1], set()).add(i)
                self.launches.append(i)
            elif w[0] == "record":
                events[w[1]] = set(streams.get(w[2], ()))
            elif w[0] == "wait":
                streams.setdefault(w[1], set()).update(events.get(w[2], ()))
            elif w[0] == "sync_event":
                host |= events.get(w[1], set())
            elif w[0] == "sync_stream":
                host |= streams.get(w[1], set())
            elif w[0] in ("sync_device", "free"):   # hipFree waits for the device
                host |= set(self.launches)
            elif w[0] == "copy" and w[2] == "1":
                self.unwaited.append([log[k] for k in self.launches if k not in host])


def build(folder):
    lib = os.path.join(str(folder), "libamdhip64.so.7")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-pthread", "-Wl,-soname,libamdhip64.so.7", "-o", lib,
                    os.path.join(HERE, "fake_hip.c")], check=True)
    return lib


def run(lib, script):
    """The script's output; its assertions fail the calling test."""
    env = dict(os.environ)
    env["LD_LIBRARY_PATH"] = os.path.dirname(lib) + ":" + env.get("LD_LIBRARY_PATH", "")
    env["PYTHONPATH"] = ":".join([HERE, os.path.join(ROOT, "gt-tomography_amd"), os.path.join(ROOT, "oracle"),
                                  env.get("PYTHONPATH", "")])
    r = subprocess.run([sys.executable, "-c", PRELUDE.format(lib=lib) + script], env=env, capture_output=True, text=True,
                       timeout=240)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
    return r.stdout

"""Builds the host code against fake_hip.cpp and loads it in place of the library."""
import ctypes as C
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "nuosc_amd", "csrc")


def build(where):
    import nuosc_amd.build as B
    out = os.path.join(str(where), "libnuosc_fake.so")
    srcs = [os.path.join(CSRC, s) for s in ("nuosc_capi.cpp", "nuosc_xfer.cpp", "vgrid.cpp")]
    subprocess.run(["g++", *B.HOST_FLAGS, "-O1", "-shared", f"-I{CSRC}", *srcs, os.path.join(ROOT, "tests", "fake_hip.cpp"),
                    "-o", out, "-lpthread"], check=True)
    return out


def load(path):
    import nuosc_amd as N
    L = C.CDLL(path)
    for name, (args, res) in N.SIGNATURES.items():
        if hasattr(L, name):
            getattr(L, name).argtypes, getattr(L, name).restype = args, res
    for name in ("count", "mistakes", "device_bytes", "graphs"):
        getattr(L, "fake_" + name).restype = C.c_longlong
    for name in ("host_flags", "event_flags"):
        getattr(L, "fake_" + name).restype = C.c_uint
    L.fake_best_zlen.argtypes = [C.c_int, C.c_double]
    return L

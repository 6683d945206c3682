"""The planner of the marching kernels (csrc/march_plans.hpp), compiled for the host by the tests that ask it."""
import ctypes as C
import functools
import os
import subprocess
import tempfile

from pv_dec_original_amd import _native as N

HERE = os.path.dirname(os.path.abspath(__file__))
CONV = ("tx", "ty", "ntx", "nty", "zseg", "nzs", "hx", "hp", "su", "nsteps", "ng", "K", "g", "roll", "rt", "wm", "wx",
        "wn", "lds")
WGRAD = ("tx", "ty", "ntx", "nty", "zseg", "nzs", "hx", "hp", "gr", "su", "fu", "cf", "ns", "nf", "units", "per",
         "splits", "lds")


@functools.lru_cache(maxsize=1)
def lib():
    with tempfile.TemporaryDirectory() as d:
        out = os.path.join(d, "libplan_probe.so")
        subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-Wall", os.path.join(HERE, "plans", "plan_probe.cpp"),
                        "-o", out], check=True)
        L = C.CDLL(out)
    L.probe_kept.restype = C.c_int64
    return L


def _plan(fn, fields, shape, cin, cout):
    out, us = (C.c_int32 * len(fields))(), C.c_double()
    got = fn(C.byref(N.NetShape(*shape)), cin, cout, out, len(fields), C.byref(us))
    return dict(zip(fields, out), us=us.value, marches=got == 2) if got else None


def conv_plan(shape, cin, cout):
    """The plan of a 3x3x3 convolution as a dict, with its price in us and whether the layer takes it, or None."""
    return _plan(lib().probe_conv_plan, CONV, shape, cin, cout)


def wgrad_plan(shape, cin, cout):
    return _plan(lib().probe_wgrad_plan, WGRAD, shape, cin, cout)


def kept(shape, cin, cout):
    """Searches so far after a lookup in the kept plans, and whether it gave the searched plan."""
    same = C.c_int32()
    n = lib().probe_kept(C.byref(N.NetShape(*shape)), cin, cout, C.byref(same))
    return n, bool(same.value)

"""The library's size rules (gcnasm_amd/csrc/routes.hpp), loaded from tests/harness/libroutes.so: what a dispatch chooses for
given sizes, without a GPU."""
import ctypes
import os
import subprocess

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "harness")
_lib = None


def lib():
    global _lib
    if _lib is None:
        path = os.path.join(HERE, "libroutes.so")
        if not os.path.exists(path):
            subprocess.check_call(["make", "-C", HERE, "libroutes.so"], stdout=subprocess.DEVNULL)
        _lib = ctypes.CDLL(path)
    return _lib


def mx_padding_in_launch(rows, k):
    return bool(lib().route_mx_padding_in_launch(ctypes.c_longlong(rows), ctypes.c_longlong(k)))

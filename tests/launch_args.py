"""hrn_args.h as a library of host code."""
import ctypes
import functools
import os
import subprocess
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))


@functools.lru_cache(None)
def library():
    with tempfile.TemporaryDirectory() as tmp:
        so = os.path.join(tmp, "launch_args.so")
        subprocess.run([os.environ.get("CXX", "g++"), "-O2", "-fPIC", "-shared", "-std=c++17", "-Wall", "-Werror", "-Wno-class-memaccess",
                        os.path.join(HERE, "launch_args_lib.cpp"), "-o", so], check=True)
        return ctypes.CDLL(so)

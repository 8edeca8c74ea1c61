"""Builds a C++ file of tests/native with the host compiler: the device code's
own headers, compiled for the CPU."""
import ctypes
import os
import subprocess

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")


def load(name, tmp):
    out = os.path.join(str(tmp), name + ".so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-Wall", "-Wno-unknown-pragmas", "-I", HERE, "-shared",
                    "-fPIC", "-o", out,
                    os.path.join(HERE, name + ".cpp")], check=True)
    return ctypes.CDLL(out)

"""Builds of the CPU emulation with other limits (test infrastructure): macros
of the kernels and of the emulation itself given on the command line, for the
paths that the usual limits keep rare."""
from __future__ import annotations

import ctypes
import os
import subprocess
from concurrent.futures import ThreadPoolExecutor

from fastlem_amd import _native

from . import build as _build

_libs = {}


def lib(name: str, source: str = "", header: str = "", **macros):
    """The library built with ``macros``, as build/libfastlem_emu_<name>.so;
    ``source`` (a file of this folder) compiled in, ``header`` included in every
    file."""
    if name not in _libs:
        out = os.path.join(os.path.dirname(_build.lib_path()), f"libfastlem_emu_{name}.so")
        os.makedirs(os.path.dirname(out), exist_ok=True)
        srcs = [os.path.join(_build.CSRC, s) for s in _build.SOURCES] + [os.path.join(_build.HERE, "emu.cpp")]
        headers = [os.path.join(_build.CSRC, h) for h in os.listdir(_build.CSRC) if h.endswith(".h")]
        srcs += [os.path.join(_build.HERE, source)] if source else []
        headers += [os.path.join(_build.HERE, header)] if header else []
        headers += [os.path.join(_build.HERE, "include", "hip", "hip_runtime.h"), os.path.abspath(__file__)]
        if not os.path.exists(out) or os.path.getmtime(out) < max(map(os.path.getmtime, srcs + headers)):
            flags = ["-std=c++17", "-O1", "-fPIC", "-pthread", "-ffp-contract=off", "-fno-fast-math",
                     "-U_FORTIFY_SOURCE", "-D_FORTIFY_SOURCE=0", "-fno-omit-frame-pointer", "-w",
                     "-I", os.path.join(_build.HERE, "include"), "-I", os.path.join(_build.ROOT, "include")]
            flags += [f"-D{k}={v}" for k, v in macros.items()]
            flags += ["-include", os.path.join(_build.HERE, header)] if header else []
            tmp = f"{out}.{os.getpid()}"  # (several processes may build it at a time)
            objects = [f"{tmp}.{os.path.basename(src)}.o" for src in srcs]

            def compile_one(src, obj):
                lang = ["-x", "c++"] if src.endswith(".hip") else []
                subprocess.run(["g++"] + flags + lang + ["-c", src, "-o", obj], check=True)

            with ThreadPoolExecutor(4) as pool:
                list(pool.map(compile_one, srcs, objects))
            subprocess.run(["g++", "-shared", "-pthread"] + objects + ["-o", tmp], check=True)
            for obj in objects:
                os.remove(obj)
            os.replace(tmp, out)
        _libs[name] = _native._declare(ctypes.CDLL(out))
    return _libs[name]

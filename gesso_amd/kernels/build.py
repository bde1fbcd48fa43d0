"""Compiling and loading the HIP extension.

The kernels under ``gesso_amd/csrc`` are compiled with ``hipcc`` for gfx950 into one shared
library with a C interface and loaded through ``ctypes``; ``host.cpp``, the launches a step makes most
without the interpreter between check and launch, becomes a Python module beside it where there is a C++
compiler with Python's and torch's headers.  Both lie in the tree
(``gesso_amd/_lib``) when that folder can be written, else in a per-user temporary folder.
A digest of the sources and flags lies beside it; a library whose digest differs is built
again.  Nothing here falls back to another implementation: if the library cannot be built
or loaded, :class:`~gesso_amd.errors.KernelError` says why.
"""
from __future__ import annotations

import ctypes
import hashlib
import importlib.util
import os
import shutil
import subprocess
import sys
import sysconfig
import tempfile
import threading
import time
from concurrent.futures import ThreadPoolExecutor

import torch

from ..errors import KernelError

ARCH = "gfx950"
CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "csrc")
LIB_NAME = "libgesso_hip.so"
# packed float32 instructions are switched off: some of their forms have given wrong results
FLAGS = ["--offload-arch=" + ARCH, "-O3", "-fPIC", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
         "-packed-fp32-ops", "-Wno-unused-command-line-argument"]

# the vendor's matrix product library (products of many rows, library_gemm.hip)
LINK = ["-lhipblaslt"]

# the module of host.cpp: compiled against the interpreter and the torch that import it
HOST_NAME = "gesso_host"
HOST_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}"]
HOST_LINK = ["-ltorch_python", "-ltorch_cpu", "-lc10", "-ldl"]
# (where these lie is not part of the digest: a tree may be built on one machine and run on another)
_TORCH = os.path.dirname(torch.__file__)
_HOST_INCLUDE = [os.path.join(_TORCH, "include"), os.path.join(_TORCH, "include", "torch", "csrc", "api", "include"),
                 sysconfig.get_paths()["include"]]

_lock = threading.Lock()
_lib = None
_host = None


def sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))


def _digest() -> str:
    h = hashlib.sha256()
    h.update(" ".join(FLAGS + LINK + HOST_FLAGS + HOST_LINK + [torch.__version__, sys.version]).encode())
    for name in sorted(os.listdir(CSRC)):
        if name.endswith((".hip", ".h", ".cpp")):
            h.update(name.encode())
            with open(os.path.join(CSRC, name), "rb") as f:
                h.update(f.read())
    return h.hexdigest()


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"),
                 os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise KernelError("hipcc not found: the HIP extension cannot be built (set HIPCC or ROCM_PATH)")


def _cxx():
    """A C++ compiler for the host module, or None."""
    for cand in (shutil.which("g++"), os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "clang++")):
        if cand and os.path.exists(cand):
            return cand
    return None


def _host_lacks():
    """What the host module cannot be compiled for want of, or None."""
    if _cxx() is None:
        return "a C++ compiler"
    for header, where in (("Python.h", _HOST_INCLUDE[-1]), ("torch/csrc/autograd/python_variable.h", _HOST_INCLUDE[0])):
        if not os.path.exists(os.path.join(where, header)):
            return header
    return None


def _lib_dirs():
    """Candidate folders for the library, the in-tree one first."""
    tree = os.path.join(os.path.dirname(CSRC), "_lib")
    user = os.path.join(tempfile.gettempdir(), f"gesso_amd_{os.getuid()}")
    return [tree, user]


def _writable(d: str) -> bool:
    try:
        os.makedirs(d, exist_ok=True)
        probe = os.path.join(d, f".probe{os.getpid()}")
        with open(probe, "w"):
            pass
        os.remove(probe)
        return True
    except OSError:
        return False


def _say(msg: str) -> None:
    print(f"[gesso_amd build] {msg}", file=sys.stderr, flush=True)


def build(force: bool = True, verbose: bool = True) -> str:
    """Compile every kernel source for gfx950 and link the library; returns its path."""
    digest = _digest()
    out_dir = next((d for d in _lib_dirs() if _writable(d)), None)
    if out_dir is None:
        raise KernelError("no writable folder for the HIP extension", tried=_lib_dirs())
    lib = os.path.join(out_dir, LIB_NAME)
    stamp = lib + ".digest"
    if not force and _is_build(lib, digest):
        return lib
    hipcc = _hipcc()
    obj_dir = os.path.join(out_dir, "obj")
    os.makedirs(obj_dir, exist_ok=True)
    srcs = sources()
    env = dict(os.environ)
    env.setdefault("HOME", out_dir)   # hipcc's helpers want some HOME
    t0 = time.time()
    if verbose:
        _say(f"compiling {len(srcs)} HIP sources for {ARCH} into {out_dir}")

    def compile_one(name):
        obj = os.path.join(obj_dir, name[:-4] + ".o")
        cmd = [hipcc] + FLAGS + ["-c", os.path.join(CSRC, name), "-o", obj]
        p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, env=env)
        if p.returncode != 0:
            raise KernelError(f"hipcc failed on {name}:\n{p.stdout[-4000:]}")
        if verbose:
            _say(f"  {name} done ({time.time() - t0:.0f} s)")
        return obj

    tmp, host_tmp = lib + f".tmp{os.getpid()}", _host_path(lib) + f".tmp{os.getpid()}"

    def compile_host():
        where = [f for d in _HOST_INCLUDE for f in ("-isystem", d)]
        p = subprocess.run([_cxx()] + HOST_FLAGS + where + ["-o", host_tmp, os.path.join(CSRC, "host.cpp"), "-L" + os.path.join(_TORCH, "lib")] + HOST_LINK,
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, env=env)
        if p.returncode != 0:
            raise KernelError(f"compiling the host module failed:\n{p.stdout[-4000:]}")
        if verbose:
            _say(f"  host.cpp done ({time.time() - t0:.0f} s)")

    lacks = _host_lacks()
    if lacks is not None:
        _say(f"no {lacks}: built without the host module, every launch is made from Python (slower steps of short prompts, the same results)")
    workers = max(1, min(len(srcs), int(os.environ.get("MAX_JOBS", "0")) or (os.cpu_count() or 4), 16))
    try:
        with ThreadPoolExecutor(workers) as pool:
            host = pool.submit(compile_host) if lacks is None else None
            objs = list(pool.map(compile_one, srcs))
            if host is not None:
                host.result()
        p = subprocess.run([hipcc, "--offload-arch=" + ARCH, "-shared", "-fPIC", "-o", tmp] + objs + LINK,
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, env=env)
        if p.returncode != 0:
            raise KernelError(f"linking the HIP extension failed:\n{p.stdout[-4000:]}")
        # library, module and digest belong together: nothing is replaced before all is made, and no digest stands beside a
        # library and a module of two builds
        if os.path.exists(stamp):
            os.remove(stamp)
        os.replace(tmp, lib)
        if host is not None:
            os.replace(host_tmp, _host_path(lib))
        elif os.path.exists(_host_path(lib)):
            os.remove(_host_path(lib))
    finally:
        for left in (tmp, host_tmp):
            if os.path.exists(left):
                os.remove(left)
    with open(stamp, "w") as f:
        f.write(digest + ("" if lacks is None else "\n" + _WITHOUT_HOST + lacks))
    if verbose:
        _say(f"built {lib} in {time.time() - t0:.0f} s")
    return lib


def _host_path(lib: str) -> str:
    return os.path.join(os.path.dirname(lib), HOST_NAME + ".so")


_WITHOUT_HOST = "without the host module for want of "           # (a digest's second line)


def _is_build(lib: str, digest: str) -> bool:
    """Whether the library there is of this digest, with its host module unless it was built without one."""
    try:
        with open(lib + ".digest") as f:
            held = f.read().strip().split("\n")
    except OSError:
        return False
    without = len(held) > 1 and held[1].startswith(_WITHOUT_HOST)
    return held[0] == digest and os.path.exists(lib) and (without or os.path.exists(_host_path(lib)))


def find_built():
    """Path of a library whose digest matches the sources, or None."""
    digest = _digest()
    return next((lib for lib in (os.path.join(d, LIB_NAME) for d in _lib_dirs()) if _is_build(lib, digest)), None)


_C_TYPES = {"int": ctypes.c_int, "long": ctypes.c_long, "float": ctypes.c_float, "double": ctypes.c_double,
            "unsigned": ctypes.c_uint}


def entry_points():
    """``name -> (result type, argument types)`` of every ``extern "C"`` entry point, read from the sources' own
    declarations: with these set, a call passes plain Python numbers and addresses and ctypes converts them by table
    instead of guessing per argument (a third of a call's cost on the host)."""
    import re
    out = {}
    pattern = re.compile(r'extern\s+"C"\s+(const char\*|int|long)\s+(gs_\w+)\s*\(([^)]*)\)\s*\{')
    for name in sorted(os.listdir(CSRC)):
        if not name.endswith((".hip", ".h")):
            continue
        with open(os.path.join(CSRC, name), encoding="utf-8") as f:
            text = f.read()
        for res, fn, args in pattern.findall(text):
            types = []
            for a in (a.strip() for a in args.split(",") if a.strip()):
                if "*" in a or a.startswith("hipStream_t"):
                    types.append(ctypes.c_void_p)
                else:
                    words = a.replace("const ", "").split()
                    if words[0] not in _C_TYPES:
                        raise KernelError(f"{name}: {fn} takes {a!r}, which the loader has no ctypes type for")
                    types.append(_C_TYPES[words[0]])
            out[fn] = (ctypes.c_char_p if "char" in res else (ctypes.c_long if res == "long" else ctypes.c_int), types)
    return out


def load_host():
    """The module of ``host.cpp``, bound to the loaded library; None where that was built without it."""
    global _host
    lib = load()
    with _lock:
        path = _host_path(lib._name)
        if _host is None and os.path.exists(path):
            try:
                spec = importlib.util.spec_from_file_location(HOST_NAME, path)
                host = importlib.util.module_from_spec(spec)
                spec.loader.exec_module(host)
                host.bind(lib._name, KernelError)
            except (ImportError, OSError) as err:
                raise KernelError(f"cannot load the host module {path}: {err}") from err
            _host = host
        return _host


def load() -> ctypes.CDLL:
    """The loaded library; built first if no current build is found."""
    global _lib
    with _lock:
        if _lib is not None:
            return _lib
        path = find_built()
        if path is None:
            path = build(force=False)
        try:
            _lib = ctypes.CDLL(path)
        except OSError as err:
            raise KernelError(f"cannot load the HIP extension {path}: {err}") from err
        for fn, (res, args) in entry_points().items():
            try:
                f = getattr(_lib, fn)
            except AttributeError:
                continue
            f.restype, f.argtypes = res, args
        _lib.gs_last_error.restype = ctypes.c_char_p
        if _lib.gs_abi_version() != 15:
            raise KernelError("the HIP extension has another interface version; build it again")
        return _lib

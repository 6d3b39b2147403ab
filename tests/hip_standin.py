"""The host side of libg4a over a stand-in for the HIP runtime
(tests/cpp/hip_standin.cpp): the library's own dispatch, workspace and capture
code on a machine without a GPU, which records the kernels a call launches."""
import ctypes
import functools
import importlib.util
import re
import subprocess
import sys
from collections import namedtuple

from g4a import build

OUT = build.REPO / "tests" / "cpp" / "_build" / "standin"
CLANG = "/opt/rocm/llvm/bin/clang++"
PTR = 0x7000_0000_0000  # an aligned "device" address for operands: nothing reads it

Launch = namedtuple("Launch", "name gx gy gz threads")


def _build():
    OUT.mkdir(parents=True, exist_ok=True)
    host, rt, lib = OUT / "g4a.o", OUT / "runtime.o", OUT / "libg4a.so"
    flags = ["-O1", "-w", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__", f"-I{build.INCLUDE}", f"-I{build.CSRC}",
             "-I/opt/rocm/include"]
    build._run([CLANG, "-x", "hip", "--cuda-host-only", *flags, "-c", build.CSRC / "g4a.cpp", "-o", host], False)
    build._run([CLANG, *flags, "-c", build.REPO / "tests" / "cpp" / "hip_standin.cpp", "-o", rt], False)
    # the device code that the host object would register
    symbols = subprocess.run(["nm", "-u", str(host)], capture_output=True, text=True, check=True).stdout
    fat = re.findall(r"\b__hip_fatbin\w*", symbols)
    build._run([CLANG, "-shared", "-Wl,-Bsymbolic", *[f"-Wl,--defsym={s}=0" for s in fat], host, rt, "-o", lib, "-ldl"],
               False)
    return lib


@functools.lru_cache(maxsize=1)
def binding():
    """A copy of the g4a package over the stand-in, beside the real one."""
    pkg = build.PKG / "g4a" / "__init__.py"
    spec = importlib.util.spec_from_file_location("g4a_on_standin", pkg, submodule_search_locations=[str(pkg.parent)])
    mod = importlib.util.module_from_spec(spec)
    sys.modules[spec.name] = mod  # (its dataclasses look their module up)
    spec.loader.exec_module(mod)
    lib = mod.load_library(_build())
    lib.standin_budget.argtypes = [ctypes.c_size_t]
    lib.standin_used.restype = ctypes.c_size_t
    lib.standin_launches.restype = ctypes.c_size_t
    lib.standin_launches.argtypes = [ctypes.c_char_p, ctypes.c_size_t]
    return mod


def budget(nbytes=None):
    """The device memory there is, in all (None: no limit)."""
    binding().load_library().standin_budget(ctypes.c_size_t(-1).value if nbytes is None else nbytes)


def used():
    return binding().load_library().standin_used()


def sync_error(code):
    binding().load_library().standin_sync_error(code)


def last_error():
    """The error the thread's next launch check would find, which this clears."""
    return binding().load_library().hipGetLastError()


def launches():
    """The launches since the last call."""
    lib = binding().load_library()
    buf = ctypes.create_string_buffer(1 << 20)
    assert lib.standin_launches(buf, len(buf)) <= len(buf)
    rows = [line.split() for line in buf.value.decode().splitlines()]
    return [Launch(r[0], *map(int, r[1:])) for r in rows]


def weight(N, K, bits, signed=False, qbytes=PTR):
    g = binding()
    return g.DeviceQWeight(g.QWeightArgs(qbytes, PTR, N, K, bits, int(signed), K), None, None)

"""Runs a test's function in a process of its own, where the library's HIP
calls go to tests/fake_hip.cpp: host code on the CPU, no GPU, no kernels.

    out = fake_hip.call(__name__, "some_function", arg, ...)

some_function(hip, pe, arg, ...) gets the fake runtime (Hip below) and the
package; what it returns comes back through JSON, and an assertion that fails
there fails the test.
"""
import ctypes
import functools
import importlib
import json
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@functools.lru_cache(maxsize=None)
def _library() -> str:
    out = os.path.join(tempfile.mkdtemp(prefix="fake_hip_"), "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I/opt/rocm/include", "-o", out,
                    os.path.join(HERE, "fake_hip.cpp")], check=True)
    return out


def call(module: str, function: str, *args):
    p = subprocess.run([sys.executable, os.path.abspath(__file__), _library(), module, function, json.dumps(args)],
                       capture_output=True, text=True, timeout=300, cwd=ROOT)
    assert p.returncode == 0, p.stderr[-3000:]
    return json.loads(p.stdout.splitlines()[-1])


class LkArgs(ctypes.Structure):
    """prism::LkArgs (csrc/gemm_lookup.hpp)."""
    _fields_ = [(n, ctypes.c_uint64) for n in ("lut", "idx", "X", "Y", "P")] + \
               [(n, ctypes.c_uint32) for n in ("M", "N", "K", "ldy", "G", "per_split", "KS")]


# Arguments of other kernels that tests look at.
PLAIN = {"k_pack_x": [("X", ctypes.c_uint64), ("Xp", ctypes.c_uint64), ("M", ctypes.c_uint32), ("K", ctypes.c_uint32),
                      ("steps", ctypes.c_uint32), ("tiles", ctypes.c_uint32)],
         "k_gemm_split_sum": [("P", ctypes.c_uint64), ("Y", ctypes.c_uint64), ("mn", ctypes.c_uint64),
                              ("S", ctypes.c_uint32)]}


class Launch:
    """One kernel launch; `lk`: the arguments of a lookup GEMM kernel, `args`: of a kernel of PLAIN."""

    def __init__(self, name, grid, threads, stream, lk, args):
        self.name, self.grid, self.threads, self.stream, self.lk, self.args = name, grid, threads, stream, lk, args


class Hip:
    def __init__(self, path):
        self.lib = lib = ctypes.CDLL(path, mode=ctypes.RTLD_GLOBAL)
        lib.fake_log_size.restype = ctypes.c_size_t
        lib.fake_log_line.restype, lib.fake_log_line.argtypes = ctypes.c_char_p, [ctypes.c_size_t]
        lib.fake_set_capturing.argtypes = [ctypes.c_void_p]
        lib.fake_refuse.argtypes = [ctypes.c_size_t]
        lib.fake_room.restype, lib.fake_room.argtypes = ctypes.c_size_t, [ctypes.c_uint64]
        self.launches, self.on_append = [], None
        kind = ctypes.CFUNCTYPE(None, ctypes.c_char_p, ctypes.POINTER(ctypes.c_uint), ctypes.POINTER(ctypes.c_void_p),
                                ctypes.c_void_p)

        def on_launch(name, dims, args, stream):
            name = name.decode()
            lk = None
            if "k_gemm_lookup" in name:
                lk = LkArgs.from_buffer_copy(ctypes.string_at(args[0], ctypes.sizeof(LkArgs)))
            plain = next((v for k, v in PLAIN.items() if k in name), [])
            values = {n: t.from_address(args[i]).value for i, (n, t) in enumerate(plain)}
            self.launches.append(Launch(name, (dims[0], dims[1]), dims[3], stream or 0, lk, values))
            if self.on_append:  # (a call's own scratch is gone once the call returns)
                self.on_append(self.launches[-1])

        self._on_launch = kind(on_launch)
        lib.fake_on_launch(self._on_launch)

    def clear(self):
        self.lib.fake_log_clear()
        self.launches.clear()

    def log(self):
        return [self.lib.fake_log_line(i).decode() for i in range(self.lib.fake_log_size())]

    def room(self, address: int) -> int:
        """Bytes from `address` to the end of its live device allocation (0: in none)."""
        return self.lib.fake_room(address)

    def malloc(self, nbytes: int) -> int:
        p = ctypes.c_void_p()
        assert self.lib.hipMalloc(ctypes.byref(p), ctypes.c_size_t(nbytes)) == 0
        return p.value


class Tensor:
    """Stands for a device tensor of `nbytes` in the package's calls."""

    def __init__(self, hip, nbytes, offset=0):
        self.n, self.address = nbytes, hip.malloc(nbytes + offset) + offset

    def data_ptr(self):
        return self.address

    def numel(self):
        return self.n

    def element_size(self):
        return 1


def _main():
    path, module, function, args = sys.argv[1:]
    hip = Hip(path)
    sys.path[:0] = [HERE, ROOT]
    pe = importlib.import_module("prism-engine_amd")
    print(json.dumps(getattr(importlib.import_module(module), function)(hip, pe, *json.loads(args))))


if __name__ == "__main__":
    _main()

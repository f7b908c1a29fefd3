"""csrc/bounds.h built by the host compiler: the arithmetic the kernels run, in
the kernels' own source, over numpy arrays."""
from __future__ import annotations

import ctypes
import functools
import subprocess
import tempfile
from pathlib import Path

import numpy as np

SHIM = Path(__file__).resolve().parent / "bounds_shim.cpp"


@functools.lru_cache(maxsize=None)
def load() -> ctypes.CDLL:
    out = Path(tempfile.mkdtemp(prefix="athx_bounds_")) / "bounds.so"
    # -ffp-contract=off, as the kernels are built.
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-fPIC", "-shared", "-Wall", "-Werror", str(SHIM),
                    "-o", str(out)], check=True)
    return ctypes.CDLL(str(out))


def call(name: str, n: int, out_dtype, *args):
    """The shim's ``name`` over n elements: arrays by pointer, ints as uint32."""
    keep = [np.ascontiguousarray(a) if isinstance(a, np.ndarray) else ctypes.c_uint32(a) for a in args]
    out = np.empty(n, out_dtype)
    fn = getattr(load(), name)
    fn.restype = None
    fn(*[a.ctypes.data_as(ctypes.c_void_p) if isinstance(a, np.ndarray) else a for a in keep], ctypes.c_uint32(n),
       out.ctypes.data_as(ctypes.c_void_p))
    return out

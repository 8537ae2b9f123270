"""The library's host-callable rules (csrc/slot_rule.hpp, csrc/bla_key.hpp) as
ctypes functions: the headers that the kernels use, compiled for the host."""
import ctypes
import functools
import os
import subprocess
import tempfile

from fractalshades_amd import build

SOURCE = r"""
#include "bla_key.hpp"
#include "slot_rule.hpp"
extern "C" {
int64_t first_slot(unsigned block, unsigned wave, unsigned blocks) { return fsg::first_slot(block, wave, blocks); }
unsigned redo_share(uint64_t unsure, unsigned waves) { return fsg::redo_share(unsure, waves); }
int slot_goes(unsigned filled, unsigned before) { return fsg::slot_goes(filled, before); }
int64_t radius_key(double r) { return fsg::radius_key(r); }
int64_t modulus_key(double q, int32_t e) { return fsg::modulus_key(q, e); }
int64_t hypot_key(double x, double y) { return fsg::hypot_key(x, y); }
}
"""


@functools.lru_cache(maxsize=None)
def load():
    with tempfile.TemporaryDirectory() as d:
        src, lib = os.path.join(d, "rules.hip"), os.path.join(d, "rules.so")
        with open(src, "w") as fh:
            fh.write(SOURCE)
        subprocess.run([build.HIPCC, "--cuda-host-only", "-O1", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off",
                        "-I", build.CSRC, src, "-o", lib], check=True, capture_output=True)
        f = ctypes.CDLL(lib)
    i64, u32, dbl = ctypes.c_int64, ctypes.c_uint32, ctypes.c_double
    for name, args, res in (("first_slot", (u32, u32, u32), i64), ("redo_share", (ctypes.c_uint64, u32), u32), ("slot_goes", (u32, u32), ctypes.c_int),
                            ("radius_key", (dbl,), i64), ("modulus_key", (dbl, ctypes.c_int32), i64),
                            ("hypot_key", (dbl, dbl), i64)):
        getattr(f, name).argtypes, getattr(f, name).restype = args, res
    return f

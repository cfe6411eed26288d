"""``csrc/gemm_rules.h``, compiled for the host: the lines that a GEMM's dispatch draws by sizes alone."""

import ctypes
import functools
import os
import subprocess
import tempfile

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pith_train_amd", "csrc", "gemm_rules.h")
SOURCE = f"""
#include "{HEADER}"
#define EXPORT extern "C" int64_t
EXPORT schedule(int64_t largest, int64_t sum, int64_t per_group, int64_t workgroups) {{ return pt::schedule_of_groups(largest, sum, per_group, workgroups); }}
EXPORT big_tile_parts(int64_t form, int64_t total, int64_t workgroups) {{ return pt::big_tile_parts((pt::Schedule)form, total, workgroups); }}
"""
FORMS = "in order", "eighths", "parts"


@functools.lru_cache(None)
def _library():
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "rules.so")
        subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-x", "c++", "-", "-o", path], input=SOURCE.encode(), check=True)
        return ctypes.CDLL(path)


def call(name, *args):
    f = getattr(_library(), name)
    f.restype, f.argtypes = ctypes.c_int64, [ctypes.c_int64] * len(args)
    return f(*args)


def schedule(blocks, per_group, workgroups=256):
    """(form, share, largest tile in shares) of a weight gradient whose groups have so many 128-row blocks."""
    cost = [b + 3 for b in blocks]  # and the change of tiles
    share = sum(cost) * per_group / workgroups
    return FORMS[call("schedule", max(cost), sum(cost), per_group, workgroups)], share, max(cost) / share

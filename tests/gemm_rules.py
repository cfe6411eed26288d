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
struct Args {{ int64_t mode, rows_a, rows_b, red, G, row_used, used_rows, b_stride_g, ldb, few_rows; }};
EXPORT small_tile_rows(int64_t mode, int64_t rows_a, int64_t rows_b, int64_t red, int64_t G, int64_t row_used, int64_t used_rows, int64_t ldb) {{
  return pt::small_tile_rows(Args{{mode, rows_a, rows_b, red, G, row_used, used_rows, rows_b * red, ldb, 0}});
}}
EXPORT streams_weights(int64_t rows_a, int64_t rows_b, int64_t red, int64_t G, int64_t row_used, int64_t used_rows, int64_t ldb, int64_t few_rows) {{
  return pt::streams_weights(Args{{1, rows_a, rows_b, red, G, row_used, used_rows, rows_b * red, ldb, few_rows}});
}}
EXPORT schedule(int64_t largest, int64_t sum, int64_t per_group, int64_t workgroups) {{ return pt::schedule_of_groups(largest, sum, per_group, workgroups); }}
EXPORT few_used_rows(int64_t rows, int64_t groups) {{ return pt::few_used_rows(rows, groups); }}
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


def m_grouped_tile_rows(rows_a, n, k, groups, used_rows=None, reduction_major=False):
    """Rows of the tiles that an m-grouped product of ``rows_a`` padded rows takes (0: the large ones).  ``used_rows``: how many
    of them count, where the launch knows which."""
    return call("small_tile_rows", 1, rows_a, n, k, groups, used_rows is not None, used_rows or 0, n if reduction_major else k)


def schedule(blocks, per_group, workgroups=256):
    """(form, share, largest tile in shares) of a weight gradient whose groups have so many 128-row blocks."""
    cost = [b + 3 for b in blocks]  # and the change of tiles
    share = sum(cost) * per_group / workgroups
    return FORMS[call("schedule", max(cost), sum(cost), per_group, workgroups)], share, max(cost) / share

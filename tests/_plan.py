"""The launch plans of the batched GEMMs (kai_batched_plan.h), asked on the host."""
import ctypes
import subprocess
import tempfile
from collections import namedtuple
from functools import lru_cache
from pathlib import Path

WIDE, TALL, HALF, HALF2, ROWS32, ROWS64, ROWS96, THIN32, THIN64, THIN96 = range(10)
NAMES = ["256x256", "256x128", "128x128", "128x128 K2", "128x32", "128x64", "128x96", "32x32", "32x64", "32x96"]
Q6_NONE, Q6_96X128, Q6_96X128_2, Q6_96X64_4, Q6_64X64_4 = range(-1, 4)
Plan = namedtuple("Plan", "id bn bm tiles_n tiles_m splits split_stages main pieces piece_stages r0 c0 rows cols rest sums")


@lru_cache(maxsize=1)
def _lib():
    folder = tempfile.mkdtemp(prefix="kai_plan_")
    so = Path(folder) / "plan.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", str(so),
                    str(Path(__file__).with_name("plan_query.cpp"))], check=True)
    lib = ctypes.CDLL(str(so))
    lib.plan_mmqh.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 3 + [ctypes.POINTER(ctypes.c_int64)]
    lib.plan_mmqh.restype = None
    lib.plan_mmq6.argtypes = [ctypes.c_int64] * 3
    return lib


def folded(qtype, n, k, m):
    """-> Plan of the folded fp16 GEMM (pieces 0: no tail; rest 0: no second launch)."""
    out = (ctypes.c_int64 * len(Plan._fields))()
    _lib().plan_mmqh(qtype, n, k, m, out)
    return Plan(*out)


def q6(n, k, m):
    return _lib().plan_mmq6(n, k, m)

"""The FFN's dispatch as the library compiles it: credit_amd/csrc/ffn_plan.hpp
built with g++ behind ctypes.  No GPU."""
import ctypes
import functools
import subprocess
import tempfile
from collections import namedtuple
from pathlib import Path

Plan = namedtuple("Plan", "big bm slices skew held")


@functools.cache
def _library():
    source = Path(__file__).resolve().parent / "cpp" / "ffn_plan_query.cpp"
    with tempfile.TemporaryDirectory() as d:
        out = Path(d) / "ffn_plan.so"
        subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", str(source),
                        "-o", str(out)], check=True)
        return ctypes.CDLL(str(out))


def gemm_plan(m, n, k, kn):
    """How C[m, n] over k runs with a [n, k] B (kn: [k, n])."""
    out = (ctypes.c_int64 * 5)()
    _library().ffn_plan_query(ctypes.c_int64(m), ctypes.c_int64(n), ctypes.c_int64(k), int(kn),
                              out)
    return Plan(bool(out[0]), out[1], out[2], out[3], bool(out[4]))


def kernel(plan):
    return ("256-tile" if plan.big else "held" if plan.held else f"ring {plan.bm}") + (
        f" split {plan.slices}" if plan.slices > 1 else "")


def products(rows, d, f, kn, train=False):
    """{product: plan} of one call: GEMM1 and GEMM2 (train: also the backward's
    du, da, dW1 and dW2, whose skew is not used)."""
    out = {"gemm1": gemm_plan(rows, f, d, kn), "gemm2": gemm_plan(rows, d, f, kn)}
    if train:
        out["du"] = gemm_plan(rows, f, d, not kn)
        out["da"] = gemm_plan(rows, d, f, not kn)
        # nn.Linear: dW1 [f, d] of a [N, K] B; [in, out]: dW1 [d, f] of a [K, N] one.
        out["dw1"] = gemm_plan(d, f, rows, True) if kn else gemm_plan(f, d, rows, False)
    return out

"""The FFN's dispatch as the library compiles it: credit_amd/csrc/ffn_plan.hpp
built with g++ behind ctypes.  No GPU."""
import ctypes
import functools
import subprocess
import tempfile
from collections import namedtuple
from pathlib import Path

Plan = namedtuple("Plan", "big bm slices skew held extra_lds")


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
    out = (ctypes.c_int64 * 6)()
    _library().ffn_plan_query(ctypes.c_int64(m), ctypes.c_int64(n), ctypes.c_int64(k), int(kn),
                              out)
    return Plan(bool(out[0]), out[1], out[2], out[3], bool(out[4]), out[5])


def kernel(plan):
    """The kernel of a plan and its K slices, for people and assertions."""
    return ("256-tile" if plan.big else "held" if plan.held else f"ring {plan.bm}") + (
        f" split {plan.slices}" if plan.slices > 1 else "")


def products(rows, d, f, kn):
    """{product: plan} of a training step: the forward's two and the recomputing
    backward's four."""
    # nn.Linear: dW1 [f, d] and dW2 [d, f] of [N, K] Bs; [in, out]: the other way
    # round, of [K, N] ones.
    dw = (((d, f), (f, d)) if kn else ((f, d), (d, f)))
    return {"gemm1": gemm_plan(rows, f, d, kn), "gemm2": gemm_plan(rows, d, f, kn),
            "du": gemm_plan(rows, f, d, not kn), "da": gemm_plan(rows, d, f, not kn),
            "dw1": gemm_plan(*dw[0], rows, kn), "dw2": gemm_plan(*dw[1], rows, kn)}

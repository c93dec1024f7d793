"""The dispatch rules of the any-width row kernels on the host
(credit_amd/csrc/row_rules.hpp).  No GPU."""
import ctypes
import shutil
import subprocess
from pathlib import Path

import pytest

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")

OPS = ("row", "softmax_fwd", "softmax_bwd", "softmax_logits_backward")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    source = Path(__file__).resolve().parent / "cpp" / "row_rules_query.cpp"
    out = tmp_path_factory.mktemp("rules") / "row_rules.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", str(source), "-o",
                    str(out)], check=True)
    return ctypes.CDLL(str(out))


@pytest.mark.parametrize("op", range(len(OPS)), ids=OPS)
def test_wide_workgroups_stream_wide_rows_only(rules, op):
    """1024 lanes to a row measured slower than 256 at these shapes, up to
    2.5 times, and faster at the wide ones."""
    def threads(rows, cols):
        return rules.row_rules_stream_threads(op, ctypes.c_int64(rows), ctypes.c_int64(cols))
    for rows in (1, 32, 256, 400, 512, 700, 1023, 1024, 4096):
        for cols in (1, 64, 1000, 1024):
            assert threads(rows, cols) == 256
    for rows in (400, 512, 700, 1023):
        assert threads(rows, 2048) == 256
    for rows in (1024, 100000):
        assert threads(rows, 262144) == 256
    for rows in (1, 128, 256):
        for cols in (8192, 65536):
            assert threads(rows, cols) == 1024
    assert threads(700, 32768) == (256 if OPS[op] == "softmax_bwd" else 1024)


def test_narrow_rows_take_the_least_work_at_any_number(rules):
    """Rows that one wave holds with a vector a lane are not given four."""
    def pick(rows, cols):
        return rules.row_rules_pick(ctypes.c_int64(rows), ctypes.c_int64(cols))
    for rows in (1, 2048, 2049, 3000, 20000, 1 << 24):
        for cols in (1, 3, 62, 256):
            assert pick(rows, cols) == 6401, (rows, cols)
    assert pick(100, 770) == 25601 and pick(16384, 770) == 6404
    assert pick(100, 4097) == 0


@pytest.mark.parametrize("op,read,held", [
    (0, [(100, 3), (2048, 7)], [(100, 8), (3000, 3), (20000, 62)]),
    (1, [(100, 3), (3000, 3), (8000, 15), (700, 62), (4096, 257)],
     [(20000, 3), (8000, 62), (100, 601), (20000, 257)]),
    (2, [(100, 3), (700, 7)], [(1500, 3), (100, 15), (700, 62)]),
    (3, [(100, 6), (1500, 14), (300, 62)], [(3000, 6), (700, 62), (100, 130)]),
    (4, [(100, 7), (1500, 15), (300, 201)], [(3000, 7), (700, 201), (100, 257)])])
def test_few_narrow_rows_run_read(rules, op, read, held):
    """Shapes that measured faster on READ, and on the kernels that hold a row."""
    for shapes, want in ((read, 1), (held, 0)):
        for rows, cols in shapes:
            assert rules.row_rules_narrow(op, ctypes.c_int64(rows), ctypes.c_int64(cols)) == want


@pytest.mark.parametrize("op,whole,chunks", [
    (0, [(8, 16384), (33, 65536), (16, 262144)], [(8, 28672), (16, 131072), (32, 65536)]),
    (1, [(1, 24580), (8, 24580), (8, 32768), (16, 28672)], [(1, 36864), (16, 131072)]),
    (2, [(8, 16384), (64, 32768)], [(8, 28672), (16, 131072)]),
    (3, [(16, 65536), (1, 32768)], [(7, 65544), (16, 131072)]),
    (4, [(16, 49160), (32, 49160), (32, 57344)], [(1, 65536), (16, 131072)]),
    (5, [(8, 16384)], [(8, 28672), (32, 65536)]),
    (6, [(16, 40960), (32, 49152)], [(8, 65536), (32, 57344)])])
def test_aligned_rows_in_chunks_where_they_gain(rules, op, whole, chunks):
    """Rows of whole vectors, by which of the two measured sooner."""
    for shapes, want in ((whole, 0), (chunks, 1)):
        for rows, cols in shapes:
            assert rules.row_rules_wide(op, ctypes.c_int64(rows), ctypes.c_int64(cols), 1) == want
    assert not rules.row_rules_wide(op, ctypes.c_int64(2049), ctypes.c_int64(200003), 0)
    assert rules.row_rules_wide(op, ctypes.c_int64(1), ctypes.c_int64(200003), 0)

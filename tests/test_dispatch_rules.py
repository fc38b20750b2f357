"""The dispatch rules of csrc/ebag_rules.h, compiled for the host, against what the kernels behind them do
(restated here address by address). No GPU."""
import ctypes
import itertools
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cti-inference-optimization_amd", "csrc")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    work = tmp_path_factory.mktemp("rules")
    (work / "rules.cpp").write_text(
        '#include "ebag_rules.h"\n'
        'extern "C" int ragged(uint64_t base, int64_t rows, int64_t row_bytes, int64_t dim, int elem) {\n'
        "  return cti::ragged_buffer_loads(base, rows, row_bytes, dim, elem);\n}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}",
                    str(work / "rules.cpp"), "-o", str(work / "rules.so")], check=True)
    lib = ctypes.CDLL(str(work / "rules.so"))
    lib.ragged.argtypes = [ctypes.c_uint64, ctypes.c_int64, ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    return lib


def _chunk_offsets(dim, elem):
    """First byte of each 16-byte chunk of a row: the last one is moved back to end with the row."""
    vec = 16 // elem
    return [min(c * vec, dim - vec) * elem for c in range((dim + vec - 1) // vec)]


def test_ragged_buffer_loads_are_aligned_and_inside_the_table(rules):
    for elem, dim, pad, first, rows in itertools.product((2, 4), range(1, 70), range(5), (0, 1, 2, 3), (1, 2, 5)):
        base, row_bytes = 4096 + first * elem, (dim + pad) * elem
        span = (rows - 1) * row_bytes + dim * elem
        allowed = False
        if dim * elem >= 16:
            starts = _chunk_offsets(dim, elem)
            loads = [r * row_bytes + c for r in range(rows) for c in starts]
            assert all(o >= 0 and o + 16 <= span for o in loads)
            beyond = [span + c for c in starts]  # what a lane past its bag reads: nothing
            allowed = base % 4 == 0 and all(o % 4 == 0 for o in loads + beyond)
        assert not rules.ragged(base, rows, row_bytes, dim, elem) or allowed, (elem, dim, pad, first, rows)
        # and it is taken wherever it may be, but for one-row tables, whose stride is no address
        if allowed and rows > 1:
            assert rules.ragged(base, rows, row_bytes, dim, elem), (elem, dim, pad, first, rows)


@pytest.mark.parametrize("dim,elem", [(100, 2), (300, 2), (50, 4), (515, 4)])
def test_ragged_buffer_offsets_stay_below_4_gib(rules, dim, elem):
    row_bytes = dim * elem
    limit = 2 ** 32
    taken = [rows for rows in range(limit // row_bytes - 4, limit // row_bytes + 4)
             if rules.ragged(4096, rows, row_bytes, dim, elem)]
    assert taken  # tables of just under 4 GiB are read through buffers ...
    for rows in taken:  # ... and no load, past its bag ones included, passes 32 bits
        assert rows * row_bytes + max(_chunk_offsets(dim, elem)) + 16 <= limit
    assert not rules.ragged(4096, limit // row_bytes + 1, row_bytes, dim, elem)

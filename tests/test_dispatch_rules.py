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
        "  return cti::ragged_buffer_loads(base, rows, row_bytes, dim, elem);\n}\n"
        'extern "C" int linear(int64_t M, int32_t N, int32_t K, int param_bytes, int64_t ws, int* splits, int* steps) {\n'
        "  const cti::LinearPlan p = cti::linear_plan(M, N, K, param_bytes, ws);\n"
        "  *splits = p.splits;\n  *steps = p.steps;\n  return p.form;\n}\n"
        'extern "C" int64_t linear_ws(int64_t M, int32_t N, int32_t K) { return cti::linear_workspace_bytes(M, N, K); }\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}",
                    str(work / "rules.cpp"), "-o", str(work / "rules.so")], check=True)
    lib = ctypes.CDLL(str(work / "rules.so"))
    lib.ragged.argtypes = [ctypes.c_uint64, ctypes.c_int64, ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    lib.linear.argtypes = [ctypes.c_int64, ctypes.c_int32, ctypes.c_int32, ctypes.c_int, ctypes.c_int64,
                           ctypes.POINTER(ctypes.c_int), ctypes.POINTER(ctypes.c_int)]
    lib.linear_ws.argtypes = [ctypes.c_int64, ctypes.c_int32, ctypes.c_int32]
    lib.linear_ws.restype = ctypes.c_int64
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


GENERAL, TILE128, TILE256, BAND = range(4)
NO_LIMIT = 2 ** 63 - 1


def _plan(rules, M, N, K, param_bytes, ws):
    splits, steps = ctypes.c_int(), ctypes.c_int()
    form = rules.linear(M, N, K, param_bytes, ws, ctypes.byref(splits), ctypes.byref(steps))
    return form, splits.value, steps.value


# (rows, outputs, K, bytes of a parameter (0: the plain Linear), us on an MI355X of: the tiles, the tiles with a
# workspace for splits of K, the band form, the band form with a workspace)
MEASURED = [
    # enough rows for a band per CU, or nearly
    (30000, 256, 3584, 2, 106, 104, 68, 68), (30000, 384, 3584, 2, 156, 154, 93, 93),
    (30000, 512, 3584, 2, 212, 206, 109, 109), (30000, 512, 3584, 4, 218, 211, 109, 108),
    (30000, 256, 896, 2, 37, 36, 24, 24), (30000, 512, 896, 2, 72, 71, 39, 40),
    (24576, 256, 640, 2, 28, 28, 17, 17), (65536, 128, 1792, 2, 86, 84, 68, 68),
    # few columns: the band form multiplies at least 256
    (16384, 128, 3584, 2, 50, 36, 55, 41), (30000, 128, 3584, 2, 51, 67, 59, 59), (512, 128, 3584, 0, 33, 17, 41, 19),
    # more than 512
    (8192, 1024, 3584, 2, 103, 101, 82, 79), (30000, 768, 3584, 2, 224, 223, 205, 205),
    (30000, 640, 3584, 0, 184, 184, 185, 182), (12288, 768, 896, 0, 31, 31, 31, 31),
    # short K: splits cost more than they give
    (16384, 512, 896, 2, 36, 35, 30, 47), (16384, 512, 256, 2, 20, 20, 18, 45), (16384, 512, 256, 0, 13, 13, 17, 42),
    (16384, 512, 3584, 2, 107, 105, 85, 82), (16384, 384, 1792, 4, 59, 58, 40, 44), (8192, 513, 896, 2, 35, 35, 36, 38),
    # few bands: only with K split
    (8192, 512, 7168, 0, 75, 75, 146, 78), (8192, 512, 7168, 2, 105, 102, 154, 82), (8192, 384, 3584, 2, 53, 60, 67, 43),
    (8192, 512, 3584, 2, 57, 55, 83, 57), (4096, 384, 3584, 0, 35, 29, 61, 31), (4096, 512, 3584, 2, 50, 36, 83, 41),
    (4096, 256, 3584, 2, 50, 25, 54, 26), (4096, 384, 7168, 2, 92, 71, 125, 43), (1024, 512, 3584, 2, 49, 19, 85, 33),
]


@pytest.mark.parametrize("M,N,K,param_bytes,tile,tile_ws,band,band_ws", MEASURED)
def test_linear_form_is_the_faster_one_as_measured(rules, M, N, K, param_bytes, tile, tile_ws, band, band_ws):
    """Within 10%: the estimates behind the choice are that far off where both forms are about as fast."""
    form, splits, _ = _plan(rules, M, N, K, param_bytes, 0)
    assert splits == 1
    assert (band if form == BAND else tile) <= 1.1 * min(tile, band)
    form, splits, _ = _plan(rules, M, N, K, param_bytes, NO_LIMIT)
    taken = (band_ws if splits > 1 else band) if form == BAND else (tile_ws if splits > 1 else tile)
    assert taken <= 1.1 * min(tile, tile_ws, band, band_ws)


def test_linear_splits_cover_k_and_fit_the_workspace(rules):
    shapes = itertools.product((1, 127, 129, 1000, 2048, 8192, 16385, 30000, 65537), (1, 127, 256, 257, 385, 513, 1024),
                               (128, 256, 896, 3584, 7168, 14336), (0, 2, 4))
    for M, N, K, param_bytes in shapes:
        full = rules.linear_ws(M, N, K)
        for ws in (0, M * N * 4, 2 * M * N * 4, 3 * M * N * 4 + 64, full, NO_LIMIT):
            form, splits, steps = _plan(rules, M, N, K, param_bytes, ws)
            assert form != GENERAL
            assert splits * M * N * 4 <= max(full, M * N * 4)
            assert splits == 1 or splits * M * N * 4 <= ws
            assert steps % 2 == 0 and (splits - 1) * steps < K // 64 <= splits * steps
            if form == BAND:  # gamma and beta have to fit the LDS kept for them
                assert 2 * param_bytes * K <= 28 * 1024
            if form == TILE256:
                assert splits == 1
        if full == 0:  # what the query says is never used
            assert _plan(rules, M, N, K, param_bytes, NO_LIMIT)[1] == 1


def test_linear_general_form_and_limits(rules):
    for K in (8, 64, 200, 3520):
        assert _plan(rules, 1000, 512, K, 2, NO_LIMIT)[0] == GENERAL
    for M, N, K in ((2 ** 24, 512, 128), (2 ** 36, 8, 2 ** 30), (1000, 2 ** 24, 128)):  # byte offsets past 2^31
        assert _plan(rules, M, N, K, 2, NO_LIMIT)[0] == GENERAL
        assert rules.linear_ws(M, N, K) == 0


def test_shapes_of_the_gpu_tests_take_the_band_form(rules):
    from test_gpu_linear import BAND_SPLIT, BAND_WHOLE

    for shapes, split in ((BAND_WHOLE, False), (BAND_SPLIT, True)):
        for rows, cols, n, sizes in shapes:
            for size in sizes:
                form, splits, _ = _plan(rules, rows, n, cols, size, NO_LIMIT)
                assert form == BAND and (splits > 1) == split, (rows, cols, n, size)
    # the captured shapes of test_gpu_graph.py
    assert _plan(rules, 8192, 512, 7168, 2, NO_LIMIT)[0] == BAND and _plan(rules, 8192, 512, 7168, 2, NO_LIMIT)[1] > 1
    assert _plan(rules, 16384, 512, 1792, 2, NO_LIMIT)[:2] == (BAND, 1)

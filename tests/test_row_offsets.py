"""The sub-chunk DGDA prefill's 32-bit row offsets (csrc/dgda_rows.h), compiled for the host and
compared with whole-number arithmetic over the strides and lengths that the kernels accept."""
import ctypes
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "maba-v2-architecture_amd", "csrc")
SC = 16


@pytest.fixture(scope="module")
def rows(tmp_path_factory):
    d = tmp_path_factory.mktemp("rows")
    src = d / "rows.cpp"
    src.write_text('#include "dgda_rows.h"\n'
                   'extern "C" uint32_t row(int left, int most, int step, int first, int lane_row, int r) {\n'
                   '  return maba::row_offset((uint32_t)(lane_row * step + first), r, step, maba::row_end(left, most, step, first));\n'
                   '}\n')
    so = d / "rows.so"
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-I", CSRC, "-o", str(so), str(src)], check=True)
    f = ctypes.CDLL(str(so)).row
    f.restype = ctypes.c_uint32
    return f


@pytest.mark.parametrize("L,stride,es", [(840_000, 640, 4), (1 << 20, 1280, 4), (1 << 30, 64, 4), (600, 1 << 20, 4),
                                         (700_000, 3840, 2), (5, (2 ** 31 - 1 - 4096) // 64, 4), (1, 128, 2), (17, 0, 4)])
def test_op_rows(rows, L, stride, es):
    """Every lane's four rows are rows of the sequence: the asked one, or the last for those past the end."""
    step = stride * es
    rng = random.Random(L)
    n = -(-L // SC)
    for sc in {0, n - 1, max(0, n - 2), n // 2, *(rng.randrange(n) for _ in range(20))}:
        left = L - 1 - sc * SC
        for first in (0, 120 * es):
            for g in range(4):
                for i in range(4):
                    assert rows(left, SC - 1, step, first, 4 * g, i) == min(4 * g + i, left) * step + first


@pytest.mark.parametrize("L,stride", [(400_000, 3840), (559_000, 3840), (600, 1 << 21), (300_000, 640), (16, (1 << 31) // 33),
                                      (5, (1 << 31) // 22), (1, (1 << 31) // 18), (1, 3840)])
def test_layer_rows(rows, L, stride):
    """The fused layer's seven rows per lane, three of them taps, up to its limit on L * stride."""
    C = 640
    stride = stride // 4 * 4
    assert (L + SC) * stride + C <= 2 ** 31 - 1
    step, first = 2 * stride, 2 * (C - 4)
    n = -(-L // SC)
    for sc in {0, n - 1, n // 2, min(1, n - 1)}:
        d = min(sc * SC, 3)
        left = L - 1 - (sc * SC - d)
        for g in range(4):
            for m in range(7):
                r = 4 * g + m - 3 + d
                got = rows(left, SC - 1 + d, step, first, 4 * g, r - 4 * g)
                if r < 0:   # replaced by the history: some row of the sequence
                    assert got % step == first and got // step <= left
                else:
                    assert got == min(r, left) * step + first

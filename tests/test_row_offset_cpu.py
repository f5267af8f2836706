"""The offsets that the blocked bf16 kernels hand to range-checked accesses (csrc/row_offset.h), over the sequence sizes the
operators take (T C < 2^30): compiled for the host and walked on the CPU."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "rwkv-infctx-trainer_amd", "csrc", "row_offset.h")


@pytest.fixture(scope="module")
def offsets(tmp_path_factory):
    where = tmp_path_factory.mktemp("row_offset")
    src, lib = str(where / "o.cpp"), str(where / "o.so")
    with open(src, "w") as f:
        f.write('#include "%s"\nextern "C" void offsets(int n, int T, int C, int c, uint32_t *out) {\n'
                "    for (int t = 0; t < n; t++) out[t] = wkv::row_offset(t, T, C, c);\n}\n" % HEADER)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", src, "-o", lib])
    f = ctypes.CDLL(lib).offsets

    def walk(n, T, C, c):
        out = np.zeros(n, dtype=np.uint32)
        f(n, T, C, c, out.ctypes.data_as(ctypes.c_void_p))
        return out
    return walk


@pytest.mark.parametrize("T", [1, 2, 17, 31, 32, 33, 63, 64, 65, 100, 127, 4095, 4097])
def test_tokens_past_the_end_are_out_of_range(offsets, T):
    """Every token of the last step's 64, at the widest sequence of T tokens and where 64 rows come to 2^30, 2^31, 2^32 bytes and
    elements: present ones lie at their place, missing ones at or beyond the range that starts at any head, in 32-bit bytes
    of two- and four-byte elements."""
    most = (((1 << 30) - 1) // T) // 64 * 64
    widths = {64, 4096, most, most - 64, 34_636_800} | {(1 << p) // rows // 64 * 64 + d for p in (30, 31, 32) for rows in (33, 63, 64) for d in (0, 64)}
    n = (T + 63) // 64 * 64
    t = np.arange(n)
    for C in sorted(w for w in widths if 0 < w <= most):
        for head in {0, C // 128, C // 64 - 1}:
            left = T * C - 64 * head
            for c in (0, 32, 60):
                at = offsets(n, T, C, c)
                for size in (2, 4):
                    bytes_, end = (at * np.uint32(size)), size * left
                    assert end < 1 << 32
                    assert (bytes_[:T].astype(np.int64) == size * (t[:T].astype(np.int64) * C + c)).all()
                    assert (bytes_[T:].astype(np.int64) >= end).all(), (C, head, c, size)
                    assert (bytes_.astype(np.int64) + 4 * size <= 1 << 32).all()      # (four elements at a time)

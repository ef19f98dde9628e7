"""Chunks of a kd-tree node in the GPU build, for nodes whose end lies near the largest
int: bounds formed by adding a chunk's size to a point's index would pass it."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
INT_MAX = 2**31 - 1
SRC = """
#include "kd_chunk.h"
extern "C" int size() { return rte::kKdChunk; }
extern "C" int chunks(int n) { return rte::kd_chunks(n); }
extern "C" void chunk(int l, int r, int i, int* out) {
  const rte::KdChunk c = rte::kd_chunk(l, r, i);
  out[0] = c.first;
  out[1] = c.count;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("kd")
    src, so = d / "chunk.cpp", d / "chunk.so"
    src.write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror",
                    "-I" + os.path.join(ROOT, "rt_entry_amd", "csrc"), str(src), "-o", str(so)],
                   check=True)
    return C.CDLL(str(so))


@pytest.mark.parametrize("l,r", [
    (0, 1), (0, 2048), (5, 2054), (0, INT_MAX), (1, INT_MAX), (INT_MAX - 1, INT_MAX),
    (INT_MAX - 2047, INT_MAX), (INT_MAX - 2048, INT_MAX), (INT_MAX - 2049, INT_MAX),
    (12345, INT_MAX - 2047), (0, INT_MAX - 2048)])
def test_chunks_cover_the_node(lib, l, r):
    size, n = lib.size(), r - l
    count = lib.chunks(n)
    assert count == -(-n // size)
    out = (C.c_int * 2)()
    for i in {0, 1, count // 2, count - 2, count - 1}:
        if 0 <= i < count:
            lib.chunk(l, r, i, out)
            assert (out[0], out[1]) == (l + i * size, min(size, n - i * size)), i

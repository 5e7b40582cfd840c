"""How a split launch shares its grid between tiles and decode rows (csrc/split_share.h, the
code that the host plan and the kernels compile), compiled for the CPU: whatever the step's mix,
each kind of work that there is gets workgroups, since nothing else computes it."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "nanokv-llm_amd", "csrc")
SOURCE = r"""
#include "split_share.h"
extern "C" int share(int n, int chunks, int tiles, int f8) {
  const nkv::SplitShare s = nkv::split_share(n, chunks, tiles, f8 != 0);
  return s.rows * 65536 + s.tiles;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not installed")
    d = tmp_path_factory.mktemp("split_share")
    src, so = d / "share.cpp", d / "share.so"
    src.write_text(SOURCE)
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-fPIC", "-shared", "-I", CSRC,
                    str(src), "-o", str(so)], check=True)
    return C.CDLL(str(so))


@pytest.mark.parametrize("f8", [0, 1])
def test_every_kind_of_work_gets_workgroups(lib, f8):
    for n in (2, 4, 8, 32, 64, 512):  # workgroups of a KV head
        for chunks in [*range(0, 41), 1000, 10 ** 6]:
            for tiles in (0, 5, 9, 90, 7000, 10 ** 6, 10 ** 8):
                if chunks == tiles == 0:
                    continue
                s = lib.share(n, chunks, tiles, f8)
                rows, left = s >> 16, s & 0xffff
                at = (n, chunks, tiles, rows, left)
                assert rows + left == n, at
                assert (rows > 0) == (chunks > 0) and (left > 0) == (tiles > 0), at

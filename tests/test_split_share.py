"""How a split launch shares its grid between tiles and decode rows (csrc/split_share.h, the
code that the host plan and the kernels compile), compiled for the CPU: whatever the step's mix,
each kind of work that there is gets workgroups, since nothing else computes it, and the decode
rows a wave for every group of KV heads and of query heads' columns."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "nanokv-llm_amd", "csrc")
SOURCE = r"""
#include "split_share.h"
extern "C" int share(int n, int chunks, int tiles, int f8, int ncg, int hp) {
  const nkv::SplitShare s = nkv::split_share(n, chunks, tiles, f8 != 0, ncg, hp);
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


def _instances(cus=256):
    """(workgroups of a KV head, KV heads, column groups, KV heads a wave) of the launches that
    stream decode rows (the others have them as tiles)."""
    for hk in (1, 2, 4, 8, 16, 64, 128):
        for g in (1, 2, 5, 16, 17, 33, 64, 65, 72, 128):
            ncg = -(-g // 16) if g > 16 else 1
            for hp in (1, 2, 4):
                if hk % hp or (hp > 1 and hp * g > 16):
                    continue
                for n in {max(1, cus * per_cu // hk) for per_cu in (1, 2)}:
                    if n > -(-ncg // (4 * hp)):
                        yield n, hk, ncg, hp


@pytest.mark.parametrize("f8", [0, 1])
def test_every_kind_of_work_gets_workgroups(lib, f8):
    for n, hk, ncg, hp in _instances():
        for chunks in [*range(0, 41), 1000, 10 ** 6]:
            for tiles in (0, 5, 9, 90, 7000, 10 ** 6, 10 ** 8):
                if chunks == tiles == 0:
                    continue
                s = lib.share(n, chunks, tiles, f8, ncg, hp)
                rows, left = s >> 16, s & 0xffff
                at = (n, hk, ncg, hp, chunks, tiles, rows, left)
                assert rows + left == n, at
                assert (rows > 0) == (chunks > 0) and (left > 0) == (tiles > 0), at
                # waves of each group of KV heads and columns
                assert chunks == 0 or 4 * rows * hk // (hk * ncg // hp) >= 1, at

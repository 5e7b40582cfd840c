"""The rules by which launches are chosen (csrc/launch_rules.h, the code that the host and the
kernels compile), compiled for the CPU. How a split launch shares its grid: whatever the step's mix,
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
#include "launch_rules.h"
extern "C" int share(int n, int chunks, int tiles, int dim, int f8, int ncg, int hp) {
  const nkv::SplitShare s =
      nkv::split_share(n, chunks, nkv::row_cost(dim, f8 != 0, ncg), tiles, ncg, hp);
  return s.rows * 65536 + s.tiles;
}
extern "C" int groups(int64_t n, int64_t total, int64_t max_q, int hk, int g, int most) {
  return nkv::plain_groups(n, total, max_q, hk, g, most, 256);
}
extern "C" int64_t tiles(int64_t n, int64_t max_q, int64_t qt) {
  return nkv::plain_tiles(n, max_q, qt);
}
extern "C" int wide(int64_t batch, int64_t hk, int64_t ncg, int64_t max_c, int64_t min_c) {
  return nkv::combine_wide(batch, hk, ncg, max_c, min_c, 2048);
}
extern "C" int fits(int64_t n_seqs, int64_t tiles, int64_t keys) {
  return nkv::split_fits(n_seqs, tiles, keys);
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not installed")
    d = tmp_path_factory.mktemp("launch_rules")
    src, so = d / "rules.cpp", d / "rules.so"
    src.write_text(SOURCE)
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-fPIC", "-shared", "-I", CSRC,
                    str(src), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    lib.groups.argtypes = [C.c_int64] * 3 + [C.c_int] * 3
    lib.tiles.argtypes, lib.tiles.restype = [C.c_int64] * 3, C.c_int64
    lib.wide.argtypes = [C.c_int64] * 5
    lib.fits.argtypes = [C.c_int64] * 3
    return lib


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
        for chunks in [*range(0, 41), 1000, 10 ** 6, 119304648, 10 ** 9]:
            for tiles in (0, 5, 9, 90, 7000, 10 ** 6, 10 ** 9):
                if chunks == tiles == 0:
                    continue
                s = lib.share(n, chunks, tiles, 128, f8, ncg, hp)
                rows, left = s >> 16, s & 0xffff
                at = (n, hk, ncg, hp, chunks, tiles, rows, left)
                assert rows + left == n, at
                assert (rows > 0) == (chunks > 0) and (left > 0) == (tiles > 0), at
                # waves of each group of KV heads and columns
                assert chunks == 0 or 4 * rows * hk // (hk * ncg // hp) >= 1, at


def test_positions_of_a_stream_that_fits_stay_within_32_bits(lib):
    """The tiles' cost, a range's end up to a range past it, and the decode rows' chunks."""
    at_limit, top = 0, 2 ** 31 - 1
    for n_seqs in (1, 7, 1000, top):
        for tiles in (1, 96, 10 ** 5, 10 ** 9, 2 ** 40, 2 ** 62):
            for bits in range(4, 36):
                for keys in (2 ** bits - 1, 2 ** bits, 2 ** bits + 1):
                    cost = max(tiles * -(-min(keys, top) // 64) * 9,
                               n_seqs * -(-min(keys, top) // 16))
                    if lib.fits(n_seqs, tiles, keys):
                        assert 2 * cost + 2 ** 20 < 2 ** 31, (n_seqs, tiles, keys)
                        at_limit += cost > 2 ** 28
                    else:  # nothing far from the limit is turned away
                        assert cost > 2 ** 29, (n_seqs, tiles, keys)
    assert at_limit > 0
    # 2000 rows of a million keys (shared blocks): within; 200000: beyond
    assert lib.fits(2000, 2100, 1 << 20) == 1 and lib.fits(200000, 200100, 1 << 20) == 0


@pytest.mark.parametrize("hk,g,mix,fastest", [
    # prompt lengths, and the row groups per wave measured fastest (within 3%)
    (8, 4, [333], 1), (8, 4, [1500], 1), (8, 4, [3000], 2), (8, 4, [2048] * 4, 2),
    (8, 4, [1000] * 6, 2), (8, 4, [4096] * 16, 3), (8, 4, [1] * 80 + [300], 1),
    (8, 4, [1] * 250 + [120], 1), (8, 4, [1] * 250 + [500], 2), (8, 8, [1] * 120 + [500] * 4, 2),
    (8, 8, [1] * 250 + [300], 2), (8, 8, [1] * 250 + [500] * 4, 3), (2, 4, [1] * 250 + [500], 1),
    (1, 24, [1300], 1), (1, 24, [2000], 2), (1, 24, [1000] * 6, 2), (4, 24, [600], 2),
    (1, 33, [600], 1), (1, 33, [900], 2), (1, 33, [2000], 2), (1, 40, [3000], 2),
    (1, 48, [600], 1), (1, 48, [900], 2), (1, 48, [1300], 2), (1, 48, [2000], 3),
    (1, 48, [1000] * 6, 3), (2, 24, [2000], 2), (1, 72, [600], 2), (1, 72, [1300], 3),
    (1, 96, [400], 2), (1, 96, [1300], 3), (1, 96, [1000] * 6, 3), (1, 128, [1500], 2),
])
@pytest.mark.parametrize("rows_known", [True, False])
def test_plain_tile_size_is_the_measured_one(lib, hk, g, mix, fastest, rows_known):
    # rows of q not known: every sequence's taken as the longest's
    total = sum(mix) if rows_known or len(set(mix)) > 1 else -1
    assert lib.groups(len(mix), total, max(mix), hk, g, 3) == fastest


def test_plain_tile_size_is_one_that_holds_a_group(lib):
    for most in (1, 2, 3):
        for g in range(1, 129 if most > 1 else 65):
            for n in (1, 5, 3000):
                for max_q in (1, 2, 100, 5000, 10 ** 6):
                    for total in (-1, n, n + max_q - 1, n * max_q):
                        rg = lib.groups(n, total, max_q, 8, g, most)
                        assert 1 <= rg <= most and 64 * rg >= g, (most, g, n, max_q, total)


@pytest.mark.parametrize("hq,hk,batch,longest,wide", [
    # the waves a row's merge measured fastest with (table rows of 256-token blocks)
    (32, 8, 1, 16000, True), (32, 8, 5, 16000, True), (8, 2, 3, 4000, True),
    (64, 1, 1, 16000, True), (64, 2, 12, 4000, True), (80, 1, 8, 4000, True),
    (16, 8, 5, 1000, False), (16, 1, 100, 1000, False), (64, 2, 32, 1000, False),
    (64, 1, 64, 4000, False), (64, 1, 100, 4000, False), (64, 2, 64, 4000, False),
    (32, 1, 100, 4000, False), (80, 1, 64, 4000, False), (80, 1, 100, 4000, False),
    (32, 8, 64, 8192, False),
])
def test_merge_waves_are_the_measured_ones(lib, hq, hk, batch, longest, wide):
    g = hq // hk
    chunks = -(-longest // 256) * 16
    assert lib.wide(batch, hk, -(-g // 16) if g > 16 else 1, chunks,
                    max(3 if batch > 2 else 4, -(-chunks // 128))) == wide


@pytest.mark.parametrize("dim,f8,ncg,best", [
    # the multiples of 2 (bf16) and 1 (fp8) twentieths of a step a chunk whose shares were measured
    # within 10% of the best share on average
    (128, 0, 1, (0.5, 2)), (128, 1, 1, (0.75, 3)), (64, 0, 1, (0.5, 2)), (64, 1, 1, (0.75, 2)),
    (256, 0, 1, (1, 2)), (256, 1, 1, (2, 3)), (128, 0, 2, (1, 3)), (128, 0, 4, (1.5, 6)),
    (128, 1, 2, (1.5, 6)), (256, 0, 2, (4, 6)), (256, 0, 4, (6, 10)), (256, 1, 4, (10, 16)),
])
def test_decode_rows_share_is_near_the_measured_best(lib, dim, f8, ncg, best):
    n, chunks, tiles = 512, 2000, 40000
    rows = lib.share(n, chunks, tiles, dim, f8, ncg, 1) >> 16
    lo, hi = (n * x / (x + tiles) for x in (chunks * m * (0.45 if f8 else 0.9) for m in best))
    assert lo - 1 <= rows <= hi + 1


def test_tiles_of_a_grid_cover_the_longest_sequence_at_an_odd_stride(lib):
    for qt in (1, 2, 16, 38, 48, 192):
        for max_q in (1, 2, 15, 16, 17, 33, 96, 500, 4096, 2 ** 31 - 1):
            need = -(-max_q // qt)
            assert lib.tiles(1, max_q, qt) == need
            for n in (2, 250):
                t = lib.tiles(n, max_q, qt)
                assert need <= t <= need + 1 and t % 2 == 1, (n, max_q, qt)

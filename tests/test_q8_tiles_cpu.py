"""The tile that each size of the Q8_0 linears' GPU tile tests takes: the dispatch's own choice (csrc/q8_tiles.hpp,
compiled here), so that a change of its costs cannot leave a tile untested."""
import ctypes
import os
import subprocess

import pytest

import test_gpu_q8_f32_tiles
import test_gpu_q8_few_rows
import test_gpu_q8_ring_tiles

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "candle-3d_amd", "csrc")


@pytest.fixture(scope="module")
def choice(tmp_path_factory):
    out = tmp_path_factory.mktemp("q8_tiles")
    src, lib = out / "tiles.cpp", out / "tiles.so"
    src.write_text('#include "q8_tiles.hpp"\n'
                   'static int pack(lux3d::Q8Tile t) { return t.rows * 10000 + t.cols * 10 + t.groups; }\n'
                   'extern "C" int f32(int64_t m, int64_t n, int64_t k) { return pack(lux3d::q8_tile_f32(m, n, k)); }\n'
                   'extern "C" int bf16(int64_t m, int64_t n, int64_t k) { return pack(lux3d::q8_tile_bf16(m, n, k)); }\n')
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", "-I", CSRC, "-o", str(lib), str(src)], check=True)
    dll = ctypes.CDLL(str(lib))

    def tile(dtype, m, n, k):
        fn = getattr(dll, dtype)
        fn.argtypes, fn.restype = [ctypes.c_int64] * 3, ctypes.c_int
        t = fn(m, n, k)
        return t // 10000, t // 10 % 1000, t % 10
    return tile


def _named(label):
    """(rows, cols, groups) of a label such as "64x128 / 2" or "128x128, two a CU"."""
    size, _, groups = label.split(",")[0].partition(" / ")
    rows, cols = size.split("x")
    return int(rows), int(cols), int(groups or 1)


@pytest.mark.parametrize("dtype,cases", [("f32", test_gpu_q8_f32_tiles.TILES), ("bf16", test_gpu_q8_ring_tiles.TILES)],
                         ids=["f32", "bf16"])
def test_tile_tests_reach_the_tiles_they_name(choice, dtype, cases):
    for label, m, n, k in cases:
        assert choice(dtype, m, n, k) == _named(label), (label, m, n, k)


def test_every_tile_is_named():
    assert {_named(c[0]) for c in test_gpu_q8_f32_tiles.TILES} == {(32, 128, 3), (64, 128, 2), (64, 128, 1), (128, 256, 1)}
    assert {_named(c[0]) for c in test_gpu_q8_ring_tiles.TILES} == \
        {(32, 128, 1), (64, 128, 1), (128, 128, 1), (160, 128, 1), (128, 256, 1), (256, 256, 1)}


def test_few_rows_sizes(choice):
    """Up to 16 rows of all but wide weights; the few-rows tests' longer ones take its four row tiles wherever the costs
    say so, which is for each k at 17 and more rows of a narrow weight."""
    for dtype in ("f32", "bf16"):
        assert all(choice(dtype, m, n, k) == (16, 16, 1) for m in (1, 16) for n in (1, 9216) for k in (64, 8192))
        for k in test_gpu_q8_few_rows.KS:
            assert all(choice(dtype, m, n, k) == (16, 16, 1) for m, n in test_gpu_q8_few_rows.SIZES if m <= 16)
            taken = {(m, n): choice(dtype, m, n, k) for m, n in test_gpu_q8_few_rows.SIZES if m > 16}
            assert all(t == (64, 16, 1) for t in taken.values()), (dtype, k, taken)
    # the row tiles are the launch's y: beyond 65535 of them another kernel takes the call
    for dtype in ("f32", "bf16"):
        assert choice(dtype, 65535 * 64, 1, 64)[1] in (16, 128, 256) and choice(dtype, 65535 * 64 + 1, 1, 64)[1] != 16

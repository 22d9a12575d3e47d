"""How a call of the fp8 GEMM is cut into tiles (csrc/gemm_plan.h), on the CPU:
the header is plain C++ and is compiled here as the library compiles it."""

import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "quail_amd", "csrc")
CUS = 256
STORE, SILU, QKV = 0, 1, 2

# epilogue -> its number, weight rows, depth and token counts that take every
# small tiling for a whole call and for the last tiles of a split one (Qwen3-4B's
# o, gate_up and qkv projections). The GPU tests run them.
TILING_CASES = {
    "store": (STORE, 2560, 4096, (1, 49, 97, 193, 385, 769, 1603, 6403, 6658, 6913, 7363, 8194, 13057,
                                  19585)),
    "silu": (SILU, 19456, 2560, (1, 49, 97, 193, 769, 1027, 1537, 1633)),
    "qkv": (QKV, 6144, 2560, (1, 82, 163, 322, 643, 2689, 2818, 3073, 3394, 5377)),
}
# bf16 calls (tokens, weight rows, depth) whose persistent workgroups walk two
# 256 x 256 tiles and more
MANY_TILES = [(2333, 19456, 384), (8191, 9728, 1280), (8000, 9728, 1024)]

WRAPPER = """
#include "gemm_plan.h"
using namespace qh;
using namespace qh::gemm_small;
extern "C" {
void plan(int epi, int M, int N, int K, int cus, int* out) {
  const Plan p = choose(epi, M, N, K, cus);
  out[0] = p.large; out[1] = p.small; out[2] = all_tiles(M, N);
}
int tilings(int epi) { return kTilings[epi]; }
void tiling(int epi, int i, int* out) { out[0] = kSmall[epi][i].rows; out[1] = kSmall[epi][i].tokens; }
void tile(int t, int M, int N, int* out) {
  tile_at(t, gemm::GROUP_M, (M + gemm::BM - 1) / gemm::BM, N / gemm::BR, out[0], out[1]);
}
int pieces(int from, int M, int N, int tokens, int rows) {
  return (int)Pieces(from, M, N, tokens, rows).count();
}
void piece(int from, int M, int N, int tokens, int rows, int t, int* out) {
  Pieces(from, M, N, tokens, rows).at(t, out[0], out[1]);
}
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    path = tmp_path_factory.mktemp("gemm_plan")
    (path / "wrap.cpp").write_text(WRAPPER)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-fPIC", "-shared", "-I", CSRC,
                    str(path / "wrap.cpp"), "-o", str(path / "wrap.so")], check=True, timeout=300)
    return ctypes.CDLL(str(path / "wrap.so"))


def _pair(call, *args):
    out = (ctypes.c_int * 3)()
    call(*args, out)
    return tuple(out)


@pytest.mark.parametrize("epi", [STORE, SILU, QKV])
@pytest.mark.parametrize("M,N", [(1, 256), (128, 512), (257, 1024), (513, 768), (1000, 1280),
                                 (1024, 512), (1025, 2560), (1300, 2560), (2303, 768), (2304, 768)])
def test_a_split_launches_every_piece_with_tokens_once_and_no_other(lib, epi, M, N):
    """Tiles `from` and up, for every `from`, as pieces of every small tiling:
    the launch is exactly the pieces that hold tokens. Pieces of none, launched
    beside them, took places that the cost model counted on."""
    tiles = [_pair(lib.tile, t, M, N)[:2] for t in range(-(-M // 256) * (N // 256))]
    for i in range(lib.tilings(epi)):
        rows, tokens, _ = _pair(lib.tiling, epi, i)
        cm, cn = 256 // tokens, 256 // rows
        for start in range(len(tiles) + 1):
            want = [(tm * cm + a, tn * cn + b) for tm, tn in tiles[start:]
                    for b in range(cn) for a in range(cm) if (tm * cm + a) * tokens < M]
            n = lib.pieces(start, M, N, tokens, rows)
            got = [_pair(lib.piece, start, M, N, tokens, rows, t)[:2] for t in range(n)]
            assert got == want, (tokens, rows, start)


def test_the_gpu_tests_sizes_take_every_tiling_whole_and_as_a_tail(lib):
    """A refit of the cost model that moves a size to another tiling fails here,
    rather than leave a kernel without a test."""
    for epilogue, (epi, N, K, sizes) in TILING_CASES.items():
        taken = set()
        for M in sizes:
            large, small, tiles = _pair(lib.plan, epi, M, N, K, CUS)
            assert large < tiles, (epilogue, M)
            taken.add((small, large > 0))
        assert taken == {(i, tail) for i in range(lib.tilings(epi)) for tail in (False, True)}, epilogue


def test_the_gpu_tests_many_tiles_are_many(lib):
    for M, N, K in MANY_TILES:
        assert _pair(lib.plan, STORE, M, N, K, CUS)[0] >= 2 * CUS, (M, N, K)


def test_a_depth_past_the_scale_rows_takes_whole_tiles(lib):
    for epi, N in ((STORE, 512), (SILU, 512), (QKV, 1536)):
        for M in (1, 17, 150, 700, 5000):
            large, _, tiles = _pair(lib.plan, epi, M, N, 256 * 128, CUS)
            assert large == tiles
            assert _pair(lib.plan, epi, M, N, 255 * 128, CUS)[0] < tiles or M > 700

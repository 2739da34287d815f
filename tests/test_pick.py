"""The rules that choose a GEMM's kernel (kern_amd/csrc/pick.h), compiled on the host: the manifest ops' copy of them
agrees, and at shapes with measured times the choice is no slower than the kernel that the same call ran on before
there was one to make."""
import ctypes
import os
import random
import re
import subprocess

import pytest

from kern_amd import build as kb
from kern_amd import manifest as mf
from kern_amd import ops

SHIM = """
#include "pick.h"
using namespace kern;
extern "C" int takes(int64_t M, int64_t m, int64_t k) { return takes_walk(M, m, k); }
extern "C" int tile(int64_t M, int64_t m, int64_t k, int* rows, int* weights, int64_t* lds) {
  double us = 0;
  const SmallTile* t = best_small_tile(M, m, k, &us);
  if (!t) return 0;
  *rows = t->rows, *weights = t->weights, *lds = small_tile_lds(*t, k);
  return 1;
}
extern "C" int tile8(int64_t m, int64_t n, int64_t k) {
  const SmallTile8* t = small_tile8(m, n, k);
  return t ? t->rows * 1000 + t->weights : 0;
}
extern "C" const char* entry(int i, int kind) {
  if (kind == 2) return i < (int)(sizeof kSmallTiles8 / sizeof *kSmallTiles8) ? kSmallTiles8[i].entry : nullptr;
  if (i >= (int)(sizeof kSmallTiles / sizeof *kSmallTiles)) return nullptr;
  return kind ? kSmallTiles[i].e4m3 : kSmallTiles[i].bf16;
}
extern "C" int gemv(int64_t M, int64_t N, int64_t K) { return gemv_row_groups(M, N, K); }
extern "C" int staged(int64_t M, int64_t N, int64_t K) { return gemv_staged(M, N, K); }
extern "C" int64_t gemv_lds(int64_t kg, int64_t, int64_t) { return gemv_row_group_lds(kg); }
extern "C" int64_t ring(int64_t M, int64_t m, int64_t k) { return dense_plan(M, m, k).ring_rows; }
"""


@pytest.fixture(scope="module")
def pick(tmp_path_factory):
    d = tmp_path_factory.mktemp("pick")
    (d / "shim.cpp").write_text(SHIM)
    csrc = os.path.join(os.path.dirname(kb.__file__), "csrc")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", f"-I{csrc}", str(d / "shim.cpp"), "-o",
                    str(d / "shim.so")], check=True)
    L = ctypes.CDLL(str(d / "shim.so"))
    L.ring.restype = L.gemv_lds.restype = ctypes.c_int64
    for f in (L.takes, L.ring, L.tile8, L.gemv, L.staged, L.gemv_lds):
        f.argtypes = [ctypes.c_int64] * 3
    L.tile.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_void_p] * 3
    return L


def tile_of(pick, M, N, K):
    r, w, lds = ctypes.c_int(), ctypes.c_int(), ctypes.c_int64()
    return (r.value, w.value, lds.value) if pick.tile(M, N, K, ctypes.byref(r), ctypes.byref(w), ctypes.byref(lds)) \
        else None


def dense_route(pick, M, N, K, out="bf16"):
    """What a dense call launches: "walk", "ring", a tile "t{rows}x{weights}", or "split"."""
    if out == "bf16" and pick.takes(M, N, K):
        return "walk"
    ring = pick.ring(M, N, K)
    return "ring" if ring == M else "split" if ring else "t%dx%d" % tile_of(pick, M, N, K)[:2]


def test_every_tile_has_an_entry(pick):
    pick.entry.restype = ctypes.c_char_p
    for kind, prefix in enumerate(("kern_mx_gemm_bf16_t", "kern_mx_gemm_e4m3_t", "kern_mx_gemm_mxfp8_t")):
        got, i = set(), 0
        while e := pick.entry(i, kind):
            got.add(e.decode())
            i += 1
        assert got == {e for e in kb.ENTRIES if e.startswith(prefix)}


def test_manifest_makes_the_same_dense_choice(pick):
    for K in (1024, 2048, 4096, 7168, 8192):
        for N in [256 * i for i in range(1, 40)] + [14336, 16384, 16640, 18432, 18688, 24576, 33024, 33280, 36864]:
            for M in (1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64):
                want = f"kern_mx_gemm_bf16_s{K // 1024}" if pick.takes(M, N, K) else \
                    "kern_mx_gemm_bf16_t%dx%d" % tile_of(pick, M, N, K)[:2]
                L = mf._small_gemm_launch(N, K, M, "tokens")
                assert L["entry"] == want, (M, N, K)
                if "_t" in want:
                    assert L["shared_mem"] == tile_of(pick, M, N, K)[2] <= 163840


# M, N, K, microseconds of the walk and of the tile that the fit picks, every weight from HBM
WALK_TIMES = [
    (4, 33280, 7168, 24.42, 32.87), (8, 35072, 7168, 25.28, 33.58), (1, 33536, 7168, 24.48, 32.58),
    (16, 9216, 7168, 10.96, 11.33), (17, 9216, 8192, 13.51, 14.94), (32, 9216, 7168, 12.99, 14.38),
    (16, 18432, 8192, 17.26, 19.67), (37, 17920, 7168, 18.85, 24.19), (64, 18432, 7168, 22.70, 26.65),
    (40, 18432, 4096, 14.37, 13.70), (16, 9216, 1024, 4.12, 4.73), (1, 4096, 1024, 3.47, 3.74),
    (64, 18432, 2048, 11.04, 11.64), (16, 7168, 8192, 10.58, 9.10), (64, 4096, 4096, 10.05, 6.53),
    (64, 2048, 8192, 15.07, 7.36), (32, 1024, 4096, 7.09, 5.03), (48, 9216, 2048, 7.51, 5.91),
    (64, 256, 1024, 5.83, 3.69), (2, 22528, 8192, 24.80, 20.10), (64, 9216, 7168, 18.35, 16.83),
    (40, 16384, 4096, 13.50, 10.93), (40, 7168, 7168, 13.01, 13.22), (8, 14336, 2048, 5.74, 5.95),
    (16, 12288, 4096, 8.74, 7.99), (32, 12288, 1024, 5.22, 4.98), (32, 9216, 4096, 9.24, 8.87),
    (48, 8192, 8192, 15.54, 14.98),
]


@pytest.mark.parametrize("M,N,K,walk,tile", WALK_TIMES)
def test_walk_where_it_is_faster(pick, M, N, K, walk, tile):
    """Up to 64 rows the walk is what every such call ran on before the tiles: the choice is within 3% of it."""
    route = dense_route(pick, M, N, K)
    assert (walk if route == "walk" else tile) <= 1.03 * walk, route


# M, N, K, microseconds of the ring alone and of the small tile or (split) ring and small tile that was taken before
RING_TIMES = [
    (388, 17664, 2048, 21.17, 29.34), (531, 13312, 10240, 64.84, 89.38), (5391, 1536, 2048, 22.42, 29.64),
    (422, 17152, 1024, 16.47, 18.77), (2237, 1024, 15872, 62.69, 71.31), (1973, 2048, 3584, 19.16, 21.65),
    (567, 5632, 7680, 34.74, 40.84), (3360, 768, 7680, 32.02, 36.81), (2394, 1024, 7680, 31.98, 36.64),
    (3235, 2560, 1536, 19.59, 21.91), (1025, 7680, 7680, 57.18, 79.54), (555, 6400, 15872, 63.8, 78.72),
    (550, 13568, 3584, 32.91, 41.54), (779, 9728, 4608, 37.74, 45.26), (305, 11776, 7680, 38.26, 45.48),
    (2, 33280, 12288, 46.14, 52.59), (6, 34048, 12800, 50.39, 57.45), (8, 35072, 8704, 36.87, 41.76),
    (1191, 7680, 512, 13.28, 15.46), (3885, 3072, 3072, 34.84, 37.59), (1813, 13312, 4608, 83.44, 96.02),
]


@pytest.mark.parametrize("out", ["bf16", "e4m3"])
@pytest.mark.parametrize("M,N,K,ring,other", RING_TIMES)
def test_ring_where_it_is_faster(pick, M, N, K, ring, other, out):
    """The ring is what every such call ran on before the tiles (these came out slower: a chip full of large tiles, K of
    a power of two less 512, a ring's last round of a few rows). Another tile or split may still be taken, unless it is
    what was measured."""
    route = dense_route(pick, M, N, K, out)
    was_split = (M, N, K) in [(1191, 7680, 512), (3885, 3072, 3072), (1813, 13312, 4608)]
    assert other > 1.03 * ring and (route != "split" if was_split else route[0] != "t"), route


# M, N, K whose gain is to stay: a tile against the ring (M > 64, or K without the walk), and ring rounds with tiles after
@pytest.mark.parametrize("M,N,K,route", [(40, 6144, 3584, "tile"), (200, 4096, 7168, "tile"), (200, 7168, 2048, "tile"),
                                         (128, 9216, 7168, "tile"), (17, 512, 512, "tile"), (1024, 9216, 7168, "split"),
                                         (2446, 3584, 1024, "split"), (1410, 6144, 1536, "split"),
                                         (2048, 9216, 7168, "split"), (1280, 9216, 7168, "ring"),
                                         (4096, 2048, 7168, "ring"), (2048, 7168, 8192, "ring")])
def test_dense_routes(pick, M, N, K, route):
    got = dense_route(pick, M, N, K, "e4m3")
    assert got == route or (route == "tile" and got[0] == "t"), got


def test_split_is_whole_blocks_and_leaves_rows(pick):
    """Over the declared range: the ring's rows are none, all, or whole blocks short of all."""
    rng = random.Random(3)
    seen = set()
    for _ in range(20000):
        M, N, K = rng.randint(1, 6000), 256 * rng.randint(1, 80), 512 * rng.randint(1, 32)
        r = pick.ring(M, N, K)
        assert r == M or (r % 128 == 0 and 0 <= r < M)
        seen.add("ring" if r == M else "split" if r else "tile")
        if r < M:
            assert tile_of(pick, M - r, N, K)[2] <= 163840
    assert seen == {"ring", "split", "tile"}


@pytest.mark.parametrize("M,N,K,large,tile", [
    (524, 7296, 960, 18.59, 23.03), (644, 5384, 960, 17.61, 19.67), (2367, 1664, 992, 18.72, 20.65),
    (2932, 976, 3840, 37.27, 40.48), (144, 18464, 2688, 30.14, 32.59), (399, 7320, 704, 14.59, 15.72),
    (3070, 792, 4992, 40.54, 44.91), (4050, 688, 4992, 40.99, 46.99)])
def test_mxfp8_large_tiles_where_they_are_faster(pick, M, N, K, large, tile):
    """kern_mx_gemm_mxfp8 is what every such call ran on before the small tiles (microseconds of both)."""
    assert tile > 1.03 * large and not pick.tile8(M, N, K)


@pytest.mark.parametrize("M,N,K,small", [(72, 9216, 7168, True), (16, 4096, 2048, True), (200, 4096, 7168, True),
                                         (500, 4096, 2048, True), (1, 16, 32, True), (1500, 4096, 7168, False),
                                         (2048, 2048, 7168, False), (4096, 2048, 7168, False), (300, 520, 2 << 20, False)])
def test_mxfp8_routes(pick, M, N, K, small):
    assert bool(pick.tile8(M, N, K)) == small


def test_gemv_counts_the_row_groups_lds(pick):
    """The rule's LDS of a row group's workgroup is the code object's static LDS, and its row groups run at once: more
    than one workgroup a CU only where two fit."""
    if not os.path.exists(ops.HSACO_PATH):
        pytest.skip("code object not built")
    notes = subprocess.run([os.path.join(kb.ROCM, "llvm", "bin", "llvm-readobj"), "--notes", ops.HSACO_PATH],
                           capture_output=True, text=True, check=True).stdout
    for kg in range(1, 17):
        block = re.search(rf"(?:(?!\.name:).)*\.name: +kern_mx_gemv_bf16_r{kg}\n", notes, re.S).group(0)
        static = int(re.findall(r"\.group_segment_fixed_size: +(\d+)", block)[-1])
        assert pick.gemv_lds(kg, 0, 0) == static
        for M in range(4, 17):
            for N in (16, 4096, 4112, 8192, 8208):
                if pick.gemv(M, N, 512 * kg):
                    assert N // 16 <= 256 * (163840 // (2 * M * 512 * kg + static)), (M, N, kg)


def test_manifest_makes_the_same_gemv_choice(pick):
    for M in range(1, 17):
        for kg in range(1, 18):
            for N in (16, 4080, 4096, 4112, 8192, 8208, 18432):
                assert bool(pick.gemv(M, N, 512 * kg)) == mf.gemv_row_groups(M, N, 512 * kg), (M, N, kg)
                assert bool(pick.staged(M, N, 512 * kg)) == mf.gemv_staged(M, N, 512 * kg), (M, N, kg)
            for N in range(18432, 80000, 1616):
                assert bool(pick.staged(M, N, 512 * kg)) == mf.gemv_staged(M, N, 512 * kg), (M, N, kg)


@pytest.mark.parametrize("M,N,K,row_groups", [(5, 8192, 7680, False), (5, 4096, 7680, True), (1, 18432, 7168, True),
                                              (8, 7168, 7680, False), (15, 8192, 2560, False), (16, 8192, 2560, False),
                                              (16, 7168, 512, False)])
def test_gemv_routes(pick, M, N, K, row_groups):
    assert bool(pick.gemv(M, N, K)) == row_groups


@pytest.mark.parametrize("M,N,K,staged,walk", [
    (4, 19312, 6144, 14.66, 18.74), (4, 19616, 5632, 15.31, 18.27), (5, 18864, 4608, 13.41, 15.88),
    (6, 19856, 6656, 17.74, 20.94), (6, 18592, 7680, 19.78, 23.17), (7, 20240, 2560, 9.55, 11.10),
    (7, 18896, 4608, 13.86, 16.00)])
def test_gemv_stages_slices_where_the_walk_is_slower(pick, M, N, K, staged, walk):
    """Slice staging is what every such call ran on before the walk had these lengths (microseconds of both)."""
    assert walk > 1.03 * staged and not pick.gemv(M, N, K) and pick.staged(M, N, K)


@pytest.mark.parametrize("K", [1024, 2048, 4096, 7168, 8192])
def test_walk_launch_of_a_saved_op_is_accepted(K):
    """A manifest op that launches the walk with its arguments as they always were (dbg, M, m, k, hb; one-dimensional
    grid, static LDS) matches the code object's metadata, and plans."""
    if not os.path.exists(ops.LIB_PATH):
        pytest.skip("library not built (python -m kern_amd.build)")
    N, entry = 9216, f"kern_mx_gemm_bf16_s{K // 1024}"
    params = ["in buffer<u8>"] * 4 + ["out buffer<bf16>", "i64", "bytes<4>", "i32", "i32", "i32"]
    with open(ops.HSACO_PATH, "rb") as f:
        img = f.read()
    sizes, n = (ctypes.c_uint32 * 32)(), ctypes.c_int()
    assert ops.lib().kern_code_object_param_sizes(img, len(img), entry.encode(), sizes, 32, ctypes.byref(n)) == 0
    assert list(sizes[:n.value]) == [8] * 6 + [4] * 4
    op = saved_walk_op(N, K, 5)
    p = ops.op_plan(op, 0, [0x1000 * (i + 1) for i in range(5)], {"tokens": 33})
    assert not p["skip"] and p["grid"] == (-(-N // 8 // 5), 1, 1) and p["shared"] == 0


def saved_walk_op(N, K, hb):
    p = ["in buffer<u8>"] * 4 + ["out buffer<bf16>"]
    return {"params": p, "impl": {"launches": [{
        "module": mf.MODULE, "entry": f"kern_mx_gemm_bf16_s{K // 1024}",
        "params": p + ["i64", "bytes<4>", "i32", "i32", "i32"], "block": [512, 1, 1], "grid": [-(-N // 8 // hb), 1, 1],
        "when": {"var": "tokens", "max": 64},
        "args": [{"param": i} for i in range(5)] + [{"i64": 0}, mf._rows("tokens"), {"i32": N}, {"i32": K},
                                                    {"i32": hb}]}]}}

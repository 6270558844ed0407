"""The plans of csrc/gemm_plan.hpp (which tiles a product takes, in which order it sums) and attention_plan.hpp, called on the host."""
import ctypes as C
import functools
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TYPES = ("f16", "bf16", "gated", "u8")
TILES = ("large", "split_large", "medium", "narrow", "halves")
CUS, WORKSPACE = 256, 32 << 20


@functools.lru_cache(None)
def _lib():
    folder = tempfile.mkdtemp()
    path = os.path.join(folder, "plan.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "llama.cu_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cxx", "gemm_plan.cpp"), "-o", path], check=True)
    lib = C.CDLL(path)
    i, w = C.c_int, C.c_long
    lib.rows.argtypes = [i, i, i, i, w, w, C.POINTER(i)]
    lib.left_sums.argtypes = [i, i, i, i, w, w, i, C.POINTER(i)]
    lib.tile_size.argtypes = [i, i, i, i, i, i, w, C.POINTER(i)]
    lib.few_rows.argtypes = [i, i, i, i, i, i, w, w, w, C.POINTER(i)]
    lib.gated_tiles.argtypes = [i, i, i, w, w]
    lib.large.argtypes = [i, i, i, i, i, w, i, C.POINTER(i)]
    lib.attention_again.argtypes = [i, i, i, w]
    lib.expert_rows.argtypes = [w, i, i, i, w]
    lib.rows.restype = lib.left_sums.restype = lib.large.restype = lib.tile_size.restype = lib.few_rows.restype = None
    os.unlink(path)
    os.rmdir(folder)
    return lib


def rows(M, K, N, n_mats=1, cus=CUS, workspace=WORKSPACE):
    """(tiles, splits)"""
    out = (C.c_int * 2)()
    _lib().rows(M, K, N, n_mats, cus, workspace, out)
    return TILES[out[0]], out[1]


def large(kind, M, K, N, n_mats=1, ragged=None, cus=CUS):
    """(columns, tiles of the first launch or 0, first column of the second or 0, its rows, its columns); ragged: rows of outputs off 16 bytes"""
    out = (C.c_int * 5)()
    _lib().large(TYPES.index(kind), M, K, N, n_mats, cus, int(N % 8 != 0 if ragged is None else ragged), out)
    return tuple(out)


def left_sums(M, K, N, u8=False, owned=True, cus=CUS, workspace=WORKSPACE):
    """(splits, step)"""
    out = (C.c_int * 2)()
    _lib().left_sums(int(u8), M, K, N, cus, workspace, int(owned), out)
    return out[0], out[1]


def tile_size(M, N, each, largest, narrowest, cus=CUS):
    """(rows, columns) of the tiles of products that leave compute units idle"""
    out = (C.c_int * 2)()
    _lib().tile_size(M, N, each, *largest, int(narrowest), cus, out)
    return tuple(out)


def few_rows(kind, M, K, N, n_mats=1, known=0, cus=CUS, workspace=WORKSPACE):
    """(splits, whether gemm_stream_kernel takes it, whether it marks its weights as read once); known: bytes of weights that a program goes through"""
    out = (C.c_int * 3)()
    _lib().few_rows(kind == "u8", kind == "bf16", M, K, N, n_mats, known, cus, workspace, out)
    return out[0], bool(out[1]), bool(out[2])


def gated_tiles(M, K, N, known=0, cus=CUS):
    """Whether a gated product of less than 160 tiles of 128x128 takes gemm_tile_kernel; known: as above"""
    return bool(_lib().gated_tiles(M, K, N, known, cus))


def scores_again(heads, n, T, cus=CUS):
    """Whether n new rows of T take the attention kernel that stores no scores."""
    return bool(_lib().attention_again(heads, n, T - n, cus))


def expert_rows(rows, experts, K, ff, cus=CUS):
    """Rows of a tile for products sorted by expert."""
    return _lib().expert_rows(rows, experts, K, ff, cus)

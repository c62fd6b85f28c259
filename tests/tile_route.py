"""The tile that a contraction of a shape is given (emc::pick_tile), for tests that say which kernel they run."""
import ctypes as C

from emc_amd._lib import lib

TILES = ("64x64", "128x128", "256x128", "256x256", "256x320")


def pad(n, to):
    return (n + to - 1) // to * to


def tile(rows, cols, na, nb):
    f = lib()["_ZN3emc9pick_tileEllii"]
    f.argtypes, f.restype = [C.c_int64, C.c_int64, C.c_int, C.c_int], C.c_int
    return TILES[f(rows, cols, na, nb)]


def logl_tile(S, I, prec, split, chunk=0):
    """Of the logits: padded rotations of a chunk by padded patterns."""
    return tile(pad(chunk or S, 256), pad(I, 256), 3 if prec == "bf16x3" else 2, 2 if split else 1)

"""Which tiles and K ranges a product takes (gemm_tiling.hpp), for tests that mean
a certain path."""

from __future__ import annotations

import ctypes as C
from typing import NamedTuple

from tests.native import build as native_build

SHARED, OWN = 1 << 25, 1 << 24  # floats of partials: gemms and gradients; forwards and 1x1 data gradients


class Tiling(NamedTuple):
    bm: int
    bn: int
    splits: int
    k_chunk: int
    full_tiles: int
    stream: int

    @property
    def kind(self) -> str:
        """"whole", "ranges", "streamed" or "rounds, then streamed" of which tiles."""
        how = "whole" if self.splits == 1 else "ranges"
        if self.stream:
            how = "rounds, then streamed" if self.full_tiles else "streamed"
        return f"{self.bm}x{self.bn} {how}"


def tiling(m: int, n: int, k: int, z: int = 1, floats: int = SHARED, wide: bool = False) -> Tiling:
    lib = C.CDLL(str(native_build.LIB))
    lib.chk_pick_tiling.argtypes = [C.c_uint64] * 5 + [C.c_int, C.POINTER(C.c_uint32)]
    lib.chk_pick_tiling.restype = None
    out = (C.c_uint32 * 6)()
    lib.chk_pick_tiling(m, n, k, z, floats, wide, out)
    return Tiling(*out)

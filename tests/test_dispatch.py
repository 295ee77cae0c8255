"""The host-side rules that choose a kernel, asked without a GPU.

Each table row is a size at which the kernels were timed on MI355X, with the
choices that came within 3 % of the fastest there (or within 0.3 us of it).
"""
import ctypes

import pytest


def rule(mangled, *argtypes):
    from rembed_amd import _lib
    fn = getattr(ctypes.CDLL(_lib.LIB_PATH), mangled)
    fn.argtypes, fn.restype = argtypes, ctypes.c_int
    return fn


# m, k, n, gated, tiles of RH_CTX_BF_TILE
W8_TILES = [
    (32768, 3072, 1024, False, {1}), (16384, 2048, 1024, False, {1}),
    (20000, 3072, 768, False, {1}), (24576, 3072, 1024, False, {1}),
    (16384, 768, 3072, False, {1}), (8192, 1024, 6144, False, {1}),
    (16384, 1024, 4096, False, {1}), (16384, 768, 2304, False, {3}),
    (5003, 768, 768, False, {3}), (1213, 768, 3072, False, {3}),
    (3896, 2048, 1024, False, {3}), (349, 3072, 768, False, {8}),
    (2048, 2048, 1024, False, {8}), (512, 1024, 4096, False, {8}),
    (512, 768, 4096, True, {8}), (1213, 768, 4096, True, {3}),
    (2048, 768, 6144, True, {3}), (16384, 768, 6144, True, {2, 10}),
    (32768, 1024, 6144, True, {1, 2, 10}), (24140, 3096, 5600, True, {1}),
]


@pytest.mark.parametrize("m,k,n,gated,good", W8_TILES)
def test_one_term_planes_tile(m, k, n, gated, good):
    pick = rule("_ZN2rh16pick_planes_tileEiiiiib", *[ctypes.c_int] * 5, ctypes.c_bool)
    assert pick(m, n, k, 1, 1, gated) in good

"""The host-side rules that choose a kernel, asked without a GPU, and the
registers that the built kernels got.

Each table row is a size at which the kernels were timed on MI355X, with the
choices that came within 3 % of the fastest there (or within 0.3 us of it).
"""
import ctypes
import struct

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


ROWS, L2, LONG = 0, 1, 2  # PoolKernel
POOLS = [
    # one long text among short ones, whose number decides
    (768, [520] + [12] * 1000, ROWS), (768, [520] + [60] * 200, ROWS),
    (768, [700] + [200] * 63, LONG), (768, [520] * 16, LONG), (768, [520], LONG),
    (768, [2048] * 16, LONG), (768, [8192, 7049], LONG), (768, [8192] + [5] * 4000, ROWS),
    (768, [900] + [400] * 99, ROWS), (768, [900] + [650] * 29, LONG),
    (768, [6000] + [60] * 399, LONG), (768, [512] * 8, ROWS), (384, [64] * 40, L2), (384, [65, 3], ROWS),
]


@pytest.mark.parametrize("h,lens,kernel", POOLS)
def test_mean_pooling_kernel(h, lens, kernel):
    pick = rule("_ZN2rh9pick_poolEiPKiiii", ctypes.c_int, ctypes.c_void_p, *[ctypes.c_int] * 3)
    cu = (ctypes.c_int * (len(lens) + 1))()
    for b, n in enumerate(lens):
        cu[b + 1] = cu[b] + n
    assert pick(h, cu, len(lens), 0, 1) == kernel
    # without the scale, and CLS pooling, never by way of the chunked kernel
    assert pick(h, cu, len(lens), 0, 0) == (LONG if kernel == LONG else ROWS)
    assert pick(h, cu, len(lens), 1, 1) == L2
    assert pick(h, cu, len(lens), 1, 0) == ROWS


def test_output_staging_grows_by_doubling():
    """Outputs that grow by 64 KiB a call up to the 8 MiB that are staged pin
    memory eight times, not at every call, and never more than they may."""
    grow = rule("_ZN2rh16staging_capacityEmmm", *[ctypes.c_size_t] * 3)
    grow.restype = ctypes.c_size_t
    most, cap, pinned = 8 << 20, 0, 0
    for need in range(1 << 16, most + 1, 1 << 16):
        if need > cap:
            cap, pinned = grow(cap, need, most), pinned + 1
        assert need <= cap <= most
    assert pinned == 8
    assert grow(0, 0, most) == grow(0, 1, most) == 1 << 16
    assert grow(0, most, most) == most and grow(5 << 20, 6 << 20, most) == most


@pytest.mark.parametrize("bytes_", [0, 1, 4095, 4096, 4097, 1 << 20])
def test_prefault_leaves_the_buffer_as_it_was(bytes_):
    """Pages are faulted in before the results exist: a call that then fails must
    not have changed a reused buffer, nor anything beside it."""
    touch = rule("_ZN2rh8prefaultEPvm", ctypes.c_void_p, ctypes.c_size_t)
    touch.restype = None
    was = bytes(i * 37 % 256 for i in range(4096)) * (bytes_ // 4096 + 2)
    buf = ctypes.create_string_buffer(was, len(was))
    touch(ctypes.addressof(buf) + 64, bytes_)
    assert buf.raw == was


def built_kernels():
    """The amdhsa metadata of every gfx950 kernel in the built library."""
    import msgpack
    from rembed_amd import _lib
    blob, out, at = open(_lib.LIB_PATH, "rb").read(), {}, 0
    while (at := blob.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        p = at + 32
        for _ in range(struct.unpack_from("<Q", blob, at + 24)[0]):
            off, size, n = struct.unpack_from("<QQQ", blob, p)
            target, p = blob[p + 24:p + 24 + n], p + 24 + n
            if b"gfx950" not in target:
                continue
            elf = blob[at + off:at + off + size]
            headers, = struct.unpack_from("<Q", elf, 32)
            each, count = struct.unpack_from("<HH", elf, 54)
            for h in range(headers, headers + each * count, each):
                kind, _, q, _, _, length, _, _ = struct.unpack_from("<IIQQQQQQ", elf, h)
                end = q + length
                while kind == 4 and q < end:  # PT_NOTE
                    nl, dl, note = struct.unpack_from("<III", elf, q)
                    d = q + 12 + (nl + 3) // 4 * 4
                    if note == 32:  # NT_AMDGPU_METADATA
                        for k in msgpack.unpackb(elf[d:d + dl])["amdhsa.kernels"]:
                            out[k[".name"]] = k
                    q = d + (dl + 3) // 4 * 4
        at += 24
    return out


# kernels that spill by design of their tile: the in-loop split, the GEMM that
# finishes LayerNorm rows and the 256x256 int8 tiles on four or eight waves
SPILL = ("gemm_bf16_kernel", "gemm_i8_ln_kernel", "gemm_i8_kernelILi256ELi256E")


def test_no_kernel_spills():
    kernels = built_kernels()
    assert len(kernels) > 100
    bad = [n for n, k in kernels.items()
           if k[".private_segment_fixed_size"] and not any(s in n for s in SPILL)]
    assert not bad, bad


def test_planes_tiles_of_two_workgroups_fit_twice():
    """512-thread planes kernels whose LDS fits a CU twice: at most 128 of a
    SIMD lane's 512 registers, two workgroups being four waves on each."""
    seen = 0
    for n, k in built_kernels().items():
        if "gemm_planes_kernel" not in n or k[".max_flat_workgroup_size"] != 512:
            continue
        if k[".group_segment_fixed_size"] <= 80 * 1024:
            seen += 1
            assert k[".vgpr_count"] <= 128, (n, k[".vgpr_count"])
    assert seen > 10

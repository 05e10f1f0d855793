"""The C-ABI library loads without a GPU and exports every symbol include/deepshift_hip.h declares;
argument validation (which happens before any HIP call) returns the documented status codes."""
import ctypes
import os
import re

import pytest

from deepshift_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "deepshift_hip.h")
TEST_HEADER = os.path.join(ROOT, "include", "deepshift_hip_test.h")


def declared_symbols(headers=(HEADER, TEST_HEADER)):
    names = set()
    for header in headers:
        text = open(header).read()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        names.update(re.findall(r"\b(ds_[a-z0-9_]+)\s*\(", text))
    return sorted(names)


def test_the_test_hook_is_not_in_the_production_header():
    assert declared_symbols((TEST_HEADER,)) == ["ds_test_fast_div", "ds_test_tune"]
    assert "ds_test_tune" not in declared_symbols((HEADER,))


def test_header_and_binding_agree():
    assert declared_symbols() == sorted(_lib.SIGNATURES)


def test_library_exports_every_declared_symbol():
    handle = ctypes.CDLL(_lib.LIB_PATH)
    for name in declared_symbols():
        assert hasattr(handle, name), name


def test_version_and_status_strings():
    L = _lib.lib()
    assert L.ds_version() >= 100
    assert L.ds_status_string(0) == b"ok"
    assert b"bits" in L.ds_status_string(-2)
    assert b"workspace" in L.ds_status_string(-4)


def test_size_queries():
    L = _lib.lib()
    # bits 4 -> 6 codes per word; N=64,K=576 -> comm 96; 64 channels = 4 tiles of 16 words
    # words [2 tiles][96][32] + negcount[64] + k table [(96+1)*6] + 16-bit codes [2*96*3 + 1][32],
    # each part padded to 256 bytes
    assert L.ds_tiled_bytes(64, 576, 4) == 2 * 96 * 32 * 4 + 256 + 2560 + (2 * 96 * 3 + 1) * 128 + 128
    # channels are padded to a multiple of 32
    assert L.ds_tiled_bytes(10, 6, 4) == 256 + 256 + 256 + (1 * 1 * 3 + 1) * 128
    # fields wider than 4 bits carry no 16-bit code section
    assert L.ds_tiled_bytes(10, 6, 5) == 256 + 256 + 256
    assert L.ds_tiled_bytes(64, 576, 7) == 0
    # cooperative launch: 25 tiles x 96 K groups on workgroups of 4 waves with >= 8 groups each -> 72
    # workgroups: their 8-byte arrival counters (padded to 256 bytes) + two partial tiles of 32 KiB each
    coop = 768 + 2 * 72 * 32768
    assert L.ds_conv2d_tiled_workspace_bytes(1, 64, 58, 58, 64, 3, 3, 1, 1, 4) == coop
    assert L.ds_conv2d_tiled_workspace_bytes(1, 64, 58, 58, 64, 3, 3, 1, 1, 4 | 0x200) == coop
    assert L.ds_conv2d_tiled_workspace_bytes(1, 64, 58, 58, 48, 3, 3, 1, 1, 4) == 0    # not 64 channels wide
    assert L.ds_conv2d_tiled_workspace_bytes(1, 64, 58, 58, 64, 3, 3, 1, 1, 5) == 0    # 5-bit fields
    assert L.ds_conv2d_workspace_bytes(1, 64, 58, 58, 64, 3, 3, 1, 1, 4) == L.ds_tiled_bytes(64, 576, 4) + coop
    assert L.ds_linear_workspace_bytes(64, 784, 512, 6) > 64 * 784 * 4


@pytest.mark.parametrize("bits,base,want", [(0, 0, -2), (7, 0, -2), (4, 1, -3), (4, -32, -3)])
def test_argument_validation_needs_no_gpu(bits, base, want):
    L = _lib.lib()
    one = ctypes.c_void_p(16)
    if base >= -31:  # packing accepts any non-positive base; the compute kernels need base >= -31
        assert L.ds_pack_i32(one, one, one, 4, 4, bits, base, None) == want
    assert L.ds_linear_i32(one, one, None, one, 4, 4, 4, bits, base, one, 1 << 20, None) == want
    assert L.ds_conv2d_i32(one, one, None, one, 1, 1, 4, 4, 1, 3, 3, 1, 1, bits, base, one, 1 << 20, None) == want


def test_invalid_sizes_and_workspace():
    L = _lib.lib()
    one = ctypes.c_void_p(16)
    assert L.ds_linear_i32(one, one, None, one, -1, 4, 4, 4, 0, one, 1 << 20, None) == -1
    assert L.ds_linear_i32(one, one, None, one, 4, 4, 4, 4, 0, None, 0, None) == -4
    assert L.ds_conv2d_i32(one, one, None, one, 1, 1, 2, 2, 1, 3, 3, 1, 1, 4, 0, one, 1 << 20, None) == -1
    assert L.ds_conv2d_i32(one, one, None, one, 1, 1, 4, 4, 1, 3, 3, 0, 1, 4, 0, one, 1 << 20, None) == -1
    assert L.ds_quantize_f32_i32(one, one, 10, 0, 16, 0, None) == -1
    assert L.ds_quantize_f32_i32(one, one, 10, 20, 20, 0, None) == -1
    assert L.ds_quantize_f32_i32(one, one, 10, 16, 16, 5, None) == -1
    # empty problems are fine and touch nothing
    assert L.ds_linear_i32(None, None, None, None, 0, 4, 4, 4, 0, one, 1 << 20, None) == 0
    assert L.ds_quantize_f32_i32(None, None, 0, 16, 16, 0, None) == 0


def test_matrix_core_entry_points_refuse_sizes_past_a_launch():
    """Rows times 256 threads stay below the 2^32 of a launch (larger inputs keep the kernels they had); an image without
    rows or columns is refused whatever its padding (an unsigned test against a negative height lets every row in)."""
    L = _lib.lib()
    one = ctypes.c_void_p(256)
    assert L.ds_mfma_input_bytes(1, 1, (1 << 24) - 1, 1, 3, 1, 4) > 0
    assert L.ds_mfma_input_bytes(1, 1, 1 << 24, 1, 3, 1, 4) == 0
    assert L.ds_mfma_input_bytes(1 << 20, 1, 32, 1, 1, 1, 1) == 0

    def prepare(H, W, ph, pw):
        return L.ds_mfma_prepare(one, 1, one, 1, 64, H, W, ph, pw, 1, 1, 0, 4, 0, 16, 16, None)

    for sizes in [(-1, 8, 4, 0), (0, 8, 4, 0), (8, -3, 0, 4), (8, 0, 0, 4), (8, 8, 1 << 29, 0), (8, 8, 0, 1 << 30)]:
        assert prepare(*sizes) == -1, sizes

    def conv(ph, pw, crop=0):
        return L.ds_mfma_conv2d(one, one, None, None, one, one, None, None, None, 1, 64, 8, 8, 64, 1, 1, 1, 1, crop, 0, 1, 1,
                                0, 14, 4, 16, 0, 16, 16, ph, pw, 4, 1, 1, 0, 0, 0, None)

    assert conv(1 << 17, 1 << 17) == -1     # a plane of more than 2^31 values
    assert conv(1 << 29, 0) == -1 and conv(0, 1 << 30) == -1 and conv(0, 0, 1 << 30) == -1


def test_matrix_core_entry_points_refuse_the_formats_that_conversions_refuse():
    L = _lib.lib()
    one = ctypes.c_void_p(256)

    def prepare(I, F, mode, x_bytes):
        return L.ds_mfma_prepare(one, 0, one, 1, 64, 8, 8, 1, 1, 3, 3, 0, x_bytes, mode, I, F, None)

    def conv(I, F, q_bytes, F_in=16):
        return L.ds_mfma_conv2d(one, one, None, None, one, one, None, None, None, 1, 64, 8, 8, 64, 1, 1, 1, 1, 0, 0, 1, 1, 0,
                                14, 4, F_in, 0, I, F, 0, 0, q_bytes, 1, 1, 0, 0, 0, None)

    for I, F, mode in [(0, 16, 0), (20, 20, 0), (16, -1, 0), (40, -16, 1), (16, 16, 2), (16, 16, -1)]:
        assert L.ds_quantize_f32_i32(one, one, 10, I, F, mode, None) == -1
        assert prepare(I, F, mode, 4) == -1, (I, F, mode)
    for I, F in [(1, 5), (5, 4), (12, -4)]:
        assert L.ds_quantize_pad_f32_i8(one, one, 1, 1, 4, 4, 0, 0, I, F, None) == -1
        assert prepare(I, F, 0, 1) == -1 and conv(I, F, 1) == -1, (I, F)
    assert prepare(3, 5, 1, 1) == -1                     # 8-bit activations are rounded, never cast
    assert conv(0, 16, 4) == -1 and conv(20, 20, 4) == -1 and conv(16, -1, 4) == -1
    assert conv(16, 16, 4, -1) == -1 and conv(16, 16, 4, 32) == -1


def test_pooled_entry_points_refuse_what_they_have_no_form_for():
    """ds_mfma_conv2d_pool and the packed call: windows past the form, results of 2 GB, formats, and, in the arrays, what the
    typed signature has no place for (sums, a residual, a matrix)."""
    import struct
    L = _lib.lib()
    one = ctypes.c_void_p(256)

    def pool(k=3, s=2, p=1, Nb=1, H=64, W=64, O=64, F_in=16, I=16, q_bytes=4, max_shift=14, out=one, q=one):
        return L.ds_mfma_conv2d_pool(one, one, None, out, q, None, None, Nb, 64, H, W, O, 1, 1, 1, 1, 1, 1, max_shift, 4, F_in, 1, I,
                                     16, 0, 0, q_bytes, 1, 1, 0, 0, 0, k, s, p, None)

    assert pool(k=0) == -1 and pool(k=-3) == -1 and pool(k=12) == -1 and pool(s=0) == -1 and pool(p=-1) == -1 and pool(p=2) == -1
    assert pool(H=1, W=64, p=0) == -1                           # no window fits
    assert pool(out=None, q=None) == -1 and pool(I=17) == -1 and pool(q_bytes=2) == -1 and pool(F_in=32) == -1
    assert pool(max_shift=15) == -1
    assert pool(Nb=9, H=1024, W=1024) == -1                     # 2.4 GB of sums

    def packed(y=0, out=256, q=0, residual=0, rows=0, H=64, k=3, s=2, p=1):
        pointers = struct.pack("=9Q", 256, 256, 0, y, out, q, 0, 0, residual)
        ints = struct.pack("=31i", 1, 64, H, 64, 64, 1, 1, 1, 1, 0, 0, 1, 1, rows, 14, 4, 16, 1, 16, 16, 0, 0, 4, 1, 1, 0, 0, 0, k, s, p)
        return L.ds_mfma_conv2d_packed(pointers, ints, None)

    assert packed(y=256, out=0) == -1 and packed(residual=256) == -1 and packed(rows=64, H=1) == -1
    assert packed(k=12) == -1 and packed(k=-1) == -1 and packed(s=0) == -1
    assert L.ds_mfma_conv2d_packed(None, b"", None) == -1 and L.ds_mfma_conv2d_packed(b"", None, None) == -1
    # the choice: no form, no gain
    assert L.ds_mfma_pool_pays(64, 3, 112, 112, 64, 7, 7, 14, 4, 3, 2, 1) == 1
    for sizes in [(0, 3, 112, 112, 64, 7, 7, 14, 4, 3, 2, 1), (64, 3, 112, 112, 64, 7, 7, 15, 4, 3, 2, 1),
                  (64, 3, 112, 112, 64, 7, 7, 14, 4, 12, 2, 1), (64, 3, 2, 2, 64, 7, 7, 14, 4, 3, 2, 0),
                  (64, 3, 1024, 1024, 64, 7, 7, 14, 4, 3, 2, 1), (64, 3, 112, 112, 0, 7, 7, 14, 4, 3, 2, 1)]:
        assert L.ds_mfma_pool_pays(*sizes) == 0, sizes


def test_error_is_raised_as_exception():
    with pytest.raises(_lib.DeepShiftError) as err:
        _lib.call("ds_quantize_f32_i32", None, None, 10, 0, 16, 0, None)
    assert err.value.status == -1

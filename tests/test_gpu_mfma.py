"""GPU: the matrix-core kernels (ds_mfma_*) against the CPU oracle, bit for bit: every mode (largest shift x width of the
activations) at the edges of its tiles -- channels, pixels, reduction blocks, taps grouped for few channels, crops -- with
activations over the whole range of their type, and the epilogue against the separate passes."""
import numpy as np
import pytest
import torch

from deepshift_amd import kernels, modules, modules_q, utils
from tests.conftest import random_codes

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _weights(rng, shape, top, ternary):
    s, sign = random_codes(rng, (shape[0], int(np.prod(shape[1:]))), max_s=top)
    s.flat[0], sign.flat[0] = top, -1
    if ternary:
        sign[rng.random(sign.shape) < 0.3] = 0
        sign.flat[0] = -1
    s, sign = s.reshape(shape), sign.reshape(shape)
    cw = utils.compress_bits(_dev(-s.astype(np.float32)), _dev(sign.astype(np.float32)))
    assert cw.max_field == top
    return s, sign, cw


def _activations(rng, shape, x_bytes, spread):
    if x_bytes == 1:
        return rng.integers(-128, 128, size=shape).astype(np.int8)
    x = rng.integers(-spread, spread, size=shape).astype(np.int32)
    if spread > 1 << 20:
        # rows with and without high digits, and the ends of the range
        x[..., : shape[-1] // 2] &= 0xfffff
        x[0] >>= 12
        x.flat[-1], x.flat[0], x.flat[x.size // 2] = 2 ** 31 - 1, -2 ** 31, -2 ** 27
    return x


# (Nb, C, H, W, O, k, stride, pad)
SHAPES = [(2, 64, 12, 12, 64, 3, 1, 1), (3, 24, 13, 9, 40, 5, 2, 2), (1, 3, 33, 31, 17, 7, 2, 3), (2, 33, 7, 9, 33, 1, 1, 0),
          (2, 9, 11, 10, 65, 3, 1, 1), (5, 7, 6, 5, 20, 2, 1, 0), (1, 130, 5, 5, 70, 3, 2, 1), (1, 1, 4, 4, 32, 3, 1, 1),
          (9, 40, 8, 8, 129, 1, 2, 0)]
MODES = [(14, 4), (11, 4), (6, 4), (5, 4), (3, 4), (1, 4), (14, 1), (31, 1), (7, 1), (3, 1), (2, 1)]


@pytest.mark.parametrize("spread", [1 << 20, 2 ** 31 - 1], ids=["low", "full"])
@pytest.mark.parametrize("top,x_bytes", MODES, ids=lambda v: str(v))
def test_convolutions_match_the_oracle(oracle, rng, top, x_bytes, spread):
    if x_bytes == 1 and spread > 1 << 20:
        pytest.skip("8-bit activations have one range")
    for i, (Nb, C, H, W, O, k, st, pad) in enumerate(SHAPES):
        print(top, x_bytes, spread, SHAPES[i], flush=True)
        s, sign, cw = _weights(rng, (O, C, k, k), top, ternary=i % 2 == 1)
        x = _activations(rng, (Nb, C, H, W), x_bytes, spread)
        bias = rng.integers(-2 ** 31, 2 ** 31 - 1, size=O).astype(np.int32)
        route = kernels.mfma_route(_dev(x), (pad, pad), cw, O, (k, k), x_bytes)
        assert route is not None
        got = kernels.mfma_conv2d(route[0], route[1], _dev(bias), O, (k, k), (st, st), route[2])
        xp = np.pad(x.astype(np.int32), ((0, 0), (0, 0), (pad, pad), (pad, pad)))
        want = oracle.conv2d(xp, -s.astype(np.int32), sign.astype(np.int32), bias, (st, st))
        np.testing.assert_array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("M,K,N", [(1, 7, 3), (63, 33, 31), (64, 64, 64), (65, 129, 70), (200, 1000, 130)])
def test_matrices_match_the_oracle(oracle, rng, M, K, N):
    for top in (14, 6, 3):
        s, sign, cw = _weights(rng, (N, K), top, ternary=False)
        x = _activations(rng, (M, K), 4, 2 ** 31 - 1)
        bias = rng.integers(-2 ** 20, 2 ** 20, size=N).astype(np.int32)
        want = oracle.linear(x, -s.astype(np.int32), sign.astype(np.int32), bias)
        got = kernels.linear(_dev(x), _dev(s), _dev(sign), _dev(bias), cw)
        np.testing.assert_array_equal(got.cpu().numpy(), want)
        # rows that start at an odd element: four-wide loads are off
        base = torch.empty(M * K + 1, dtype=torch.int32, device=DEV)
        base[1:] = _dev(x).reshape(-1)
        route = kernels.mfma_route(base[1:].view(M, K), 0, cw, N, (1, 1), 4)
        got = kernels.mfma_conv2d(route[0], route[1], _dev(bias), N, (1, 1), 1, route[2])
        np.testing.assert_array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("M,K,N", [(1, 7, 3), (63, 33, 31), (64, 64, 64), (65, 129, 70), (130, 1001, 33)])
def test_8_bit_matrices_match_the_oracle(oracle, rng, M, K, N):
    """Bytes are read as bytes, at any address, four times as many to a word as the other sources have: rows, columns and
    channels at the edges of 64, 32 and 4, and the prepared bytes themselves against those of the same values from float."""
    for top in (14, 3):
        s, sign, cw = _weights(rng, (N, K), top, ternary=False)
        x = _activations(rng, (M, K), 1, 128)
        want = oracle.linear(x.astype(np.int32), -s.astype(np.int32), sign.astype(np.int32), None)
        base = torch.empty(M * K + 1, dtype=torch.int8, device=DEV)
        base[1:] = _dev(x).reshape(-1)
        blob = kernels._mfma_of(cw, top, 1, N, K, 1, 1)
        floats = kernels.mfma_prepare(_dev(x).clamp(max=96).float() / 32, 0, (1, 1), 1, 3, 5)
        same = kernels.mfma_prepare(_dev(x).clamp(max=96), 0, (1, 1), 1)
        used = (M + 63) // 64 * ((K + 31) // 32) * 64 * 32
        assert torch.equal(same.data[:used], floats.data[:used])
        for xd in (_dev(x), base[1:].view(M, K)):
            prepared = kernels.mfma_prepare(xd, 0, (1, 1), 1)
            got = kernels.mfma_conv2d(prepared, blob, None, N, (1, 1), 1, top)
            np.testing.assert_array_equal(got.cpu().numpy(), want)


def test_more_blocks_of_channels_than_a_launch_has_workgroups_along_y():
    """A row of 2^16 + 3 blocks of 32 channels x 128 pixels: a workgroup of the layout pass takes several of them."""
    blocks = (1 << 16) + 3
    x = torch.randint(-128, 128, (1, blocks * 32 - 5, 1, 128), dtype=torch.int8, device=DEV)
    got = kernels.mfma_prepare(x, 0, (1, 1), 1)
    want = torch.zeros(blocks * 32, 128, dtype=torch.int8, device=DEV)
    want[:-5] = x[0, :, 0]
    want = want.view(blocks, 32, 128).transpose(1, 2).reshape(-1)
    assert torch.equal(got.data[:want.numel()].view(torch.int8), want)


@pytest.mark.parametrize("x_bytes", [4, 1])
@pytest.mark.parametrize("Nb,C,H,O,k,st", [(2, 32, 14, 40, 3, 1), (1, 64, 7, 96, 1, 1), (40, 32, 28, 64, 3, 2)])
def test_epilogue_matches_the_separate_passes(rng, x_bytes, Nb, C, H, O, k, st):
    pad = k // 2
    F_in, spec = (16, ((1, 1), 16, 16, torch.int32)) if x_bytes == 4 else (5, ((1, 1), 3, 5, torch.int8))
    s, sign, cw = _weights(rng, (O, C, k, k), 14, ternary=False)
    x = _dev(_activations(rng, (Nb, C, H, H), x_bytes, 1 << 18))
    prepared, blob, top = kernels.mfma_route(x, (pad, pad), cw, O, (k, k), x_bytes)
    y = kernels.mfma_conv2d(prepared, blob, None, O, (k, k), (st, st), top)
    scale, shift = (torch.rand(O, device=DEV) + 0.5), torch.randn(O, device=DEV)
    for residual in (None, torch.randn(y.shape, device=DEV)):
        for relu in (False, True):
            want = kernels.requantize_affine_pad(y, F_in, scale, shift, residual, relu, *spec[:3], True, spec[3])
            cache = {}
            for q_cache in (None, cache, cache):
                out, q = kernels.mfma_conv2d(prepared, blob, None, O, (k, k), (st, st), top, 0, F_in, scale, shift, residual,
                                             relu, spec, True, q_cache)
                assert torch.equal(out, want[0]) and torch.equal(q, want[1])
                del q


def test_a_cropped_window_reads_the_centre(oracle, rng):
    """A 1 x 1 convolution on the tensor that was padded for a 3 x 3."""
    s, sign, cw = _weights(rng, (64, 64, 1, 1), 14, ternary=False)
    x = _activations(rng, (3, 64, 9, 9), 4, 1 << 24)
    xp = np.pad(x, ((0, 0), (0, 0), (1, 1), (1, 1)))
    blob = kernels._mfma_of(cw, 14, 4, 64, 64, 1, 1)
    got = kernels.mfma_conv2d(kernels.mfma_prepare(_dev(xp), 0, (3, 3), 4), blob, None, 64, (1, 1), (2, 2), 14, (1, 1))
    want = oracle.conv2d(x, -s.astype(np.int32), sign.astype(np.int32), None, (2, 2))
    np.testing.assert_array_equal(got.cpu().numpy(), want)


def test_layers_without_a_form_keep_their_kernels(oracle, rng):
    """Shifts past 14 on int32 activations, left shifts: the plane and two-instruction kernels."""
    for top in (15, 20):
        s, sign, cw = _weights(rng, (64, 64, 3, 3), top, ternary=False)
        assert kernels.mfma_shift(cw, 4) is None and kernels.mfma_shift(cw, 1) == top
        x = _activations(rng, (1, 64, 6, 6), 4, 1 << 24)
        got = kernels.conv2d(_dev(x), _dev(s), _dev(sign), None, cw, 1, 1)
        xp = np.pad(x, ((0, 0), (0, 0), (1, 1), (1, 1)))
        np.testing.assert_array_equal(got.cpu().numpy(), oracle.conv2d(xp, -s.astype(np.int32), sign.astype(np.int32), None,
                                                                       (1, 1)))
    assert kernels.mfma_shift(utils.ConcWeight(None, -2, 4, max_field=3), 4) is None
    assert kernels.mfma_shift(utils.ConcWeight(None, 0, 4), 4) is None


@pytest.mark.parametrize("I,F", [(16, 16), (3, 5)])
def test_modules_match_the_float_path(I, F):
    """A plain module against its float form on values of the layer's grid small enough for float32 sums to be exact."""
    torch.manual_seed(0)
    layer = modules.Conv2dShift(20, 36, 3, padding=1, use_kernel=True, act_integer_bits=I, act_fraction_bits=F).to(DEV)
    layer.shift.data = torch.randint(-3, 1, layer.shift.shape, device=DEV).float()
    layer.sign.data = torch.randint(0, 2, layer.sign.shape, device=DEV).float() * 2 - 1
    layer.bias.data.zero_()
    x = torch.randint(-3, 4, (2, 20, 9, 9), device=DEV).float()
    with torch.no_grad():
        want = torch.nn.functional.conv2d(x, layer.sign * 2.0 ** layer.shift, padding=1)
        assert torch.equal(layer(x), want)


@pytest.mark.parametrize("I,F", [(16, 16), (3, 5)])
@pytest.mark.parametrize("C,O,k,scale_up", [(32, 40, 3, 1.0), (32, 40, 3, 4000.0), (24, 16, 3, 1.0), (20, 130, 1, 4000.0)])
def test_operands_from_the_epilogue_equal_the_padded_tensor(rng, I, F, C, O, k, scale_up):
    """The hand-off in the operand layout: what it holds, and what the next layer makes of it, twice into the same buffer
    (flags of the first pass must not survive), over values with and without digits 3 and 4."""
    x_bytes, dtype = (4, torch.int32) if I + F > 8 else (1, torch.int8)
    pad = k // 2
    s, sign, cw = _weights(rng, (O, C, k, k), 14, ternary=False)
    _, _, cw2 = _weights(rng, (48, O, 3, 3), 14, ternary=False)
    assert kernels.mfma_takes_prepared(cw2, 48, O, (3, 3), x_bytes)
    blob2 = kernels._mfma_of(cw2, 14, x_bytes, 48, O, 3, 3)
    cache = {}
    for H, amp in ((14, scale_up), (14, 1.0), (9, scale_up)):
        x = _dev(_activations(rng, (3, C, H, H), x_bytes, 1 << 17))
        prepared, blob, top = kernels.mfma_route(x, (pad, pad), cw, O, (k, k), x_bytes)
        scale = (torch.rand(O, device=DEV) + 0.5) * amp
        shift = torch.randn(O, device=DEV)
        args = (prepared, blob, None, O, (k, k), (1, 1), top, 0, F, scale, shift, None, False)
        _, want = kernels.mfma_conv2d(*args, ((1, 1), I, F, dtype), False)
        out, got = kernels.mfma_conv2d(*args, ((1, 1), I, F, dtype, (3, 3)), True, cache)
        assert isinstance(got, kernels.Prepared) and torch.equal(got.padded(), want)
        if x_bytes == 4 and amp > 1:
            assert bool((want.abs() >= 1 << 21).any())
        y2 = kernels.mfma_conv2d(got, blob2, None, 48, (3, 3), (2, 2), 14)
        again = kernels.mfma_conv2d(kernels.mfma_prepare(want, 0, (3, 3), x_bytes), blob2, None, 48, (3, 3), (2, 2), 14)
        assert torch.equal(y2, again)
        assert len(cache) == 1
        del got


def test_operand_buffers_are_not_reused_while_held(rng):
    s, sign, cw = _weights(rng, (32, 32, 1, 1), 3, ternary=False)
    prepared, blob, top = kernels.mfma_route(_dev(_activations(rng, (2, 32, 6, 6), 4, 1 << 17)), 0, cw, 32, (1, 1), 4)
    cache = {}
    args = (prepared, blob, None, 32, (1, 1), (1, 1), top, 0, 16, None, None, None, False, ((1, 1), 16, 16, torch.int32, (3, 3)),
            False, cache)
    first = kernels.mfma_conv2d(*args)[1]
    second = kernels.mfma_conv2d(*args)[1]
    assert first.data.data_ptr() != second.data.data_ptr()
    held = second.data.data_ptr()
    del second
    assert kernels.mfma_conv2d(*args)[1].data.data_ptr() == held


@pytest.mark.parametrize("K", [2050, 2112])
@pytest.mark.parametrize("rounded", [False, True], ids=["cast", "round"])
def test_float_matrices_match_the_oracle(oracle, rng, K, rounded):
    """The route of large LinearShift / LinearShiftQ layers: float rows converted on the way in, from an odd address, a
    row count past a block of 64, an odd row length (no four-wide loads) and one of fours, ReLU, values past the format,
    infinities and NaN."""
    M, N, I, F = 70, 45, 16, 16
    cls = modules_q.LinearShiftQ if rounded else modules.LinearShift
    layer = cls(K, N, use_kernel=True).to(DEV)
    s, sign = random_codes(rng, (N, K), max_s=14)
    with torch.no_grad():
        if rounded:
            layer.weight.copy_(_dev((sign * 2.0 ** -s).astype(np.float32)))
        else:
            layer.shift.copy_(_dev(-s.astype(np.float32)))
            layer.sign.copy_(_dev(sign.astype(np.float32)))
        layer.bias.copy_(torch.randn(N))
    x = (rng.standard_normal((M, K)) * 2.0 ** rng.integers(-18, 18, size=(M, K))).astype(np.float32)
    x.flat[::97] = np.float32("nan")
    x.flat[5::89] = np.float32("inf")
    x.flat[7::83] = -np.float32("inf")
    x.flat[11::79] = -0.0
    x.flat[13::71] = 1e-40
    x[3] = 0.25                         # a row without any of these
    base = torch.empty(M * K + 1, device=DEV)
    base[1:] = _dev(x).reshape(-1)
    convert = (lambda v: oracle.quantize(v, I, F)) if rounded else (lambda v: oracle.cast(v, F))
    bias = convert(layer.bias.detach().cpu().numpy())
    want = oracle.linear(convert(x), -s.astype(np.int32), sign.astype(np.int32), bias).astype(np.float32) / np.float32(2.0 ** F)
    with torch.no_grad():
        for xd in (_dev(x), base[1:].view(M, K)):
            np.testing.assert_array_equal(layer(xd).cpu().numpy(), want)
        np.testing.assert_array_equal(layer._kernel_forward(_dev(x), relu=True).cpu().numpy(), np.maximum(want, 0))


# (parts of the reduction, x_bytes, C, O, pixels): tiles of 32 x 64 past the fill of the chip's wave slots at which the
# reduction is one wave's (9 blocks: a quarter), and, int32 activations, between one and two tiles a slot, where two waves
# share a long one (36 blocks).  Pixel counts end inside a tile, channels inside a tile of 32 and, where the tiles of 32
# are odd in number, inside a pair of them.
LARGE = [(1, 4, 20, 70, (29, 7, 667)), (1, 4, 20, 20, (9, 1, 4789)), (1, 1, 20, 70, (31, 9, 709)), (1, 1, 120, 33, (13, 9, 877)),
         (2, 4, 120, 40, (13, 9, 667)), (2, 4, 120, 20, (19, 9, 803))]


@pytest.mark.parametrize("parts,x_bytes,C,O,pixels", LARGE, ids=lambda v: str(v).replace(" ", ""))
@pytest.mark.parametrize("top", [14, 6, 2])
def test_epilogues_of_large_launches(oracle, rng, parts, x_bytes, C, O, pixels, top):
    """The register epilogue of launches with many tiles, and the one that two waves share: sums against the oracle; float,
    padded and operand-layout results, with and without residual, against the separate passes."""
    Nb, H, W = pixels
    k, P = 3, Nb * H * W
    waves = 256 * (12 if x_bytes == 1 else 8)
    tiles = -(-O // 32) * -(-P // 64)
    fill, long = tiles / waves, C > 64
    assert P % 64 and (1 < fill < 2 and long and x_bytes == 4 if parts == 2 else fill > (1 if long else 0.25))
    s, sign, cw = _weights(rng, (O, C, k, k), top, ternary=True)
    x = _activations(rng, (Nb, C, H, W), x_bytes, 1 << 18)
    if x_bytes == 4:
        x[-1, ..., -1] = -2 ** 31           # high digits in the last tile
    bias = rng.integers(-2 ** 20, 2 ** 20, size=O).astype(np.int32)
    prepared, blob, shift_top = kernels.mfma_route(_dev(x), 1, cw, O, (k, k), x_bytes)
    y = kernels.mfma_conv2d(prepared, blob, _dev(bias), O, (k, k), 1, shift_top)
    xp = np.pad(x.astype(np.int32), ((0, 0), (0, 0), (1, 1), (1, 1)))
    want = oracle.conv2d(xp, -s.astype(np.int32), sign.astype(np.int32), bias, (1, 1), nthreads=16)
    np.testing.assert_array_equal(y.cpu().numpy(), want)
    F_in, I, F, dtype = (16, 16, 16, torch.int32) if x_bytes == 4 else (5, 3, 5, torch.int8)
    scale, shift = (torch.rand(O, device=DEV) + 0.5), torch.randn(O, device=DEV)
    for residual in (None, torch.randn(y.shape, device=DEV)):
        f, q = kernels.requantize_affine_pad(y, F_in, scale, shift, residual, True, (1, 1), I, F, True, dtype)
        args = (prepared, blob, _dev(bias), O, (k, k), 1, shift_top, 0, F_in, scale, shift, residual, True)
        out, padded = kernels.mfma_conv2d(*args, ((1, 1), I, F, dtype), True)
        assert torch.equal(out, f) and torch.equal(padded, q)
        out, handed = kernels.mfma_conv2d(*args, ((1, 1), I, F, dtype, (3, 3)), True)
        assert torch.equal(out, f) and torch.equal(handed.padded(), q)
        only, handed = kernels.mfma_conv2d(*args, ((1, 1), I, F, dtype, (3, 3)), False)
        assert only is None and torch.equal(handed.padded(), q)


@pytest.mark.parametrize("top,x_bytes", [(14, 4), (6, 4), (3, 4), (14, 1), (3, 1)], ids=lambda v: str(v))
@pytest.mark.parametrize("blocks", [1, 2, 3, 4, 5])
def test_short_reductions_of_every_digit(oracle, rng, top, x_bytes, blocks):
    """The two-set loop over odd and even numbers of blocks and the one-set loop of digit 3: channels at the edges of one
    and two tiles of 32, activations with no digit past d2, with d3 alone, with d4, and with all of them by row."""
    for N in (31, 32, 33, 64, 65):
        C = blocks * 32 - (N & 1) * 5
        s, sign, cw = _weights(rng, (N, C, 1, 1), top, ternary=N == 33)
        bias = rng.integers(-2 ** 20, 2 ** 20, size=N).astype(np.int32)
        for spread in (1 << 20, 1 << 26, 2 ** 31 - 1) if x_bytes == 4 else (128,):
            x = rng.integers(-spread, spread, size=(2, C, 5, 9)).astype(np.int32 if x_bytes == 4 else np.int8)
            if spread == 2 ** 31 - 1:
                x[:, :, 1] >>= 5
                x[:, :, 2:4] >>= 12
            prepared, blob, at = kernels.mfma_route(_dev(x), 0, cw, N, (1, 1), x_bytes)
            got = kernels.mfma_conv2d(prepared, blob, _dev(bias), N, (1, 1), 1, at)
            want = oracle.conv2d(x.astype(np.int32), -s.astype(np.int32), sign.astype(np.int32), bias, (1, 1))
            np.testing.assert_array_equal(got.cpu().numpy(), want)


# (Nb, C, H, W, k): rows of one to several workgroup's shares -- many short rows in one workgroup, the last one not full,
# parts of 32-channel blocks that fill 256 threads or just miss them, rows that take two goes
LAYOUTS = [(3, 16, 7, 5, 3), (1, 3, 9, 83, 3), (2, 40, 3, 128, 1), (1, 33, 2, 129, 1), (1, 100, 3, 41, 1), (1, 8, 2, 255, 3), (1, 8, 2, 254, 3),
           (1, 2, 2, 600, 3), (1, 70, 2, 300, 1)]


@pytest.mark.parametrize("x_bytes", [4, 1])
@pytest.mark.parametrize("Nb,C,H,W,k", LAYOUTS, ids=lambda v: str(v))
def test_the_layout_pass_at_the_edges_of_its_workgroups(oracle, rng, x_bytes, Nb, C, H, W, k):
    """Rows with digit d3 alone, with d4 and with neither side by side, from float, int32 or int8 images."""
    s, sign, cw = _weights(rng, (33, C, k, k), 6, ternary=False)
    x = _activations(rng, (Nb, C, H, W), x_bytes, 2 ** 31 - 1)
    if x_bytes == 4:
        x[:, :, 0] >>= 12
        x[..., W // 3:, 1] >>= 5
    pad = k // 2
    xp = np.pad(x.astype(np.int32), ((0, 0), (0, 0), (pad, pad), (pad, pad)))
    want = oracle.conv2d(xp, -s.astype(np.int32), sign.astype(np.int32), None, (1, 1))
    F = 16 if x_bytes == 4 else 5
    exact = np.float32(x) == x       # values that a float holds
    for source in (x, np.where(exact, x, 0).astype(np.float32) / np.float32(2.0 ** F)):
        if source.dtype == np.float32 and not exact.all():
            xf = np.pad(np.where(exact, x, 0).astype(np.int32), ((0, 0), (0, 0), (pad, pad), (pad, pad)))
            xf = np.clip(xf, -2 ** 31, (2 ** 15 - 1) * 2 ** 16)
            want = oracle.conv2d(xf, -s.astype(np.int32), sign.astype(np.int32), None, (1, 1))
        I, Fb = (16, 16) if x_bytes == 4 else (3, 5)
        route = kernels.mfma_route(_dev(source), (pad, pad), cw, 33, (k, k), x_bytes, I, Fb)
        got = kernels.mfma_conv2d(route[0], route[1], None, 33, (k, k), 1, route[2])
        if source.dtype == np.float32 and x_bytes == 1:
            xf = np.pad(np.clip(x.astype(np.int32), -128, 96), ((0, 0), (0, 0), (pad, pad), (pad, pad)))
            want = oracle.conv2d(xf, -s.astype(np.int32), sign.astype(np.int32), None, (1, 1))
        np.testing.assert_array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("C,O,k", [(16, 16, 3), (16, 4, 2), (8, 16, 3), (7, 16, 3), (3, 16, 5), (16, 16, 1), (15, 16, 2)])
def test_few_channels_agree_on_both_kernels(rng, C, O, k):
    """Layers of at most 16 channels around the number of terms from which the matrix cores take them: as the public entry
    points route them against the general kernels, and handed from layer to layer."""
    s, sign, cw = _weights(rng, (O, C, k, k), 14, ternary=False)
    x = _dev(_activations(rng, (5, C, 9, 11), 4, 2 ** 31 - 1))
    got = kernels.conv2d(x, _dev(s), _dev(sign), None, cw, 1, k // 2)
    xp = torch.nn.functional.pad(x, (k // 2,) * 4)
    want = kernels.conv2d_tiled(xp, kernels._tiled_of(cw, O, C, k, k), None, O, (k, k), 1, kernels.kernel_bits(cw))
    assert torch.equal(got, want)
    serves = kernels._mfma_conv_serves(5, C, xp.shape[2], xp.shape[3], O, (k, k), 1)
    assert serves == (C * k * k >= 64)
    assert kernels.mfma_takes_prepared(cw, O, C, (k, k), 4) == (serves and C > 8)
    if not serves or C <= 8:
        return
    _, _, before = _weights(rng, (C, 24, 3, 3), 14, ternary=False)
    prepared, blob, top = kernels.mfma_route(_dev(_activations(rng, (5, 24, 9, 11), 4, 1 << 18)), 1, before, C, (3, 3), 4)
    scale, shift = torch.full((C,), 40.0, device=DEV), torch.randn(C, device=DEV)
    args = (prepared, blob, None, C, (3, 3), (1, 1), top, 0, 16, scale, shift, None, False)
    pads = (k // 2, k // 2)
    padded = kernels.mfma_conv2d(*args, (pads, 16, 16, torch.int32), False)[1]
    handed = kernels.mfma_conv2d(*args, (pads, 16, 16, torch.int32, (k, k)), False)[1]
    assert torch.equal(handed.padded(), padded)
    blob = kernels._mfma_of(cw, 14, 4, O, C, k, k)
    assert torch.equal(kernels.mfma_conv2d(handed, blob, None, O, (k, k), 1, 14),
                       kernels.conv2d_tiled(padded, kernels._tiled_of(cw, O, C, k, k), None, O, (k, k), 1, kernels.kernel_bits(cw)))


@pytest.mark.parametrize("C,k", [(4, 3), (8, 2), (9, 2), (1, 6), (32, 1), (33, 1), (40, 1)])
@pytest.mark.parametrize("O", [24, 70])
def test_short_unpadded_reductions_agree_on_both_routes(monkeypatch, oracle, rng, C, k, O):
    """32 to 40 terms without padding, with and without the layout pass, whichever the rule takes: strides, an input whose
    channels are not in order in memory, the whole range of activations."""
    s, sign, cw = _weights(rng, (O, C, k, k), 14, ternary=True)
    x = _activations(rng, (3, C, 11, 13), 4, 2 ** 31 - 1)
    bias = rng.integers(-2 ** 20, 2 ** 20, size=O).astype(np.int32)
    xd = _dev(x)
    for stride in ((1, 1), (2, 1)):
        want = oracle.conv2d(x, -s.astype(np.int32), sign.astype(np.int32), bias, stride)
        for layout in (True, False):
            monkeypatch.setattr(kernels, "_layout_pass_pays", lambda *args, v=layout: v)
            for at in (xd, xd.to(memory_format=torch.channels_last), xd.transpose(2, 3).contiguous().transpose(2, 3)):
                got = kernels.conv2d(at, _dev(s), _dev(sign), _dev(bias), cw, stride, 0)
                np.testing.assert_array_equal(got.cpu().numpy(), want)


# (Nb, C, H, W, O, k, stride, pad), (pool kernel, stride, padding)
POOLED = [((2, 3, 45, 37, 64, 7, 2, 3), (3, 2, 1)), ((3, 20, 14, 9, 70, 3, 1, 1), (2, 2, 0)), ((1, 64, 9, 12, 33, 1, 1, 0), (3, 1, 1)),
          ((2, 8, 23, 23, 129, 3, 1, 1), (11, 4, 5)), ((40, 3, 64, 64, 40, 3, 2, 1), (3, 2, 0)), ((1, 33, 5, 70, 34, 3, 1, 1), (5, 3, 2)),
          ((130, 32, 8, 8, 64, 3, 1, 1), (8, 8, 0))]


@pytest.mark.parametrize("top,x_bytes", [(14, 4), (6, 4), (3, 4), (14, 1), (3, 1)], ids=lambda v: str(v))
@pytest.mark.parametrize("shape,pool", POOLED, ids=lambda v: str(v).replace(" ", ""))
def test_pooling_in_the_launch_matches_the_separate_pass(rng, top, x_bytes, shape, pool):
    """The fused max pooling against the sums and the pooling pass: windows that overlap and do not, rectangles past the
    image's edges, scales of both signs, zero and NaN, activations with digits 3 and 4 and results with them."""
    Nb, C, H, W, O, k, st, pad = shape
    s, sign, cw = _weights(rng, (O, C, k, k), top, ternary=True)
    x = _activations(rng, (Nb, C, H, W), x_bytes, 1 << 18)
    if x_bytes == 4:
        x[0, :, : H // 2] <<= 5            # d3
        x[-1, :, H - 1, W - 1] = -2 ** 31  # d4
    bias = _dev(rng.integers(-2 ** 20, 2 ** 20, size=O).astype(np.int32))
    prepared, blob, at = kernels.mfma_route(_dev(x), pad, cw, O, (k, k), x_bytes)
    F_in, I, F, dtype = (16, 16, 16, torch.int32) if x_bytes == 4 else (5, 3, 5, torch.int8)
    y = kernels.mfma_conv2d(prepared, blob, bias, O, (k, k), st, at)
    assert kernels.mfma_pool_serves(Nb, y.shape[2], y.shape[3], O, pool)
    scale, shift = torch.randn(O, device=DEV), torch.randn(O, device=DEV)
    scale[1], scale[2], shift[3] = 0.0, float("nan"), float("nan")
    for relu in (True, False):
        f, q = kernels.requantize_affine_maxpool(y, F_in, scale, shift, relu, pool, (1, 1), I, F, True, dtype)
        args = (prepared, blob, bias, O, (k, k), st, at, 0, F_in, scale, shift, None, relu)
        cache = {}
        for filt in ((3, 3), (3, 3), None):
            out, got = kernels.mfma_conv2d(*args, ((1, 1), I, F, dtype, filt), True, cache, pool)
            assert torch.equal(torch.nan_to_num(out, nan=7.0), torch.nan_to_num(f, nan=7.0))
            assert torch.equal(got.padded() if filt else got, q)
            del got
        out, _ = kernels.mfma_conv2d(*args, None, True, None, pool)
        assert torch.equal(torch.nan_to_num(out, nan=7.0), torch.nan_to_num(f, nan=7.0))
        _, got = kernels.mfma_conv2d(*args, ((0, 1), I, F, dtype, (1, 3)), False, None, pool)
        assert torch.equal(got.padded(), q[:, :, 1:-1])


@pytest.mark.parametrize("shape,pool", [((3, 16, 21, 40, 40), (2, 2, 0)), ((2, 16, 9, 131, 129), (3, 1, 1)), ((5, 16, 70, 1, 64), (1, 1, 0)),
                                        ((1, 16, 80, 12, 80), (5, 1, 2))], ids=lambda v: str(v).replace(" ", ""))
def test_each_flag_of_a_pooled_hand_off_says_what_its_values_have(rng, shape, pool):
    """Digits d3 and d4 in few places: waves whose windows lie in one flag's 32 pixels, in several, and in none that is set;
    each flag is that of its pixels and channels, no other's."""
    Nb, C, H, W, O = shape
    s, sign, cw = _weights(rng, (O, C, 1, 1), 14, ternary=False)
    x = rng.integers(-2 ** 8, 2 ** 8, size=(Nb, C, H, W)).astype(np.int32)
    for top in (2 ** 19, 2 ** 26):
        x[rng.integers(0, Nb, 3), :, rng.integers(0, H, 3), rng.integers(0, W, 3)] = rng.integers(-top, top, size=(3, C))
    prepared, blob, at = kernels.mfma_route(_dev(x), 0, cw, O, (1, 1), 4)
    scale, shift = torch.ones(O, device=DEV), torch.zeros(O, device=DEV)
    scale[::3] = 4
    y = kernels.mfma_conv2d(prepared, blob, None, O, (1, 1), 1, at)
    _, q = kernels.requantize_affine_maxpool(y, 16, scale, shift, True, pool, (1, 1), 16, 16, False, torch.int32)
    _, got = kernels.mfma_conv2d(prepared, blob, None, O, (1, 1), 1, at, 0, 16, scale, shift, None, True,
                                 ((1, 1), 16, 16, torch.int32, (3, 3)), False, None, pool)
    assert torch.equal(got.padded(), q)
    c16, pixels = (O + 15) // 16, Nb * (q.shape[2] - 2) * (q.shape[3] - 2)
    level = (q >= 2 ** 20).to(torch.uint8) + 2 * (q >= 2 ** 27 - 2 ** 20).to(torch.uint8)
    level = level[:, :, 1:-1, 1:-1].permute(0, 2, 3, 1).reshape(pixels, O)
    level = torch.nn.functional.pad(level, (0, c16 * 16 - O, 0, -pixels % 32)).view(-1, 32, c16, 16)
    want = level.amax((1, 3))
    assert 0 < int((want > 0).sum()) < want.numel() and int(want.max()) == 3
    planes = (q.shape[0] * q.shape[2] * q.shape[3] * ((O + 31) // 32 * 32) * 5 + 64 + 255) // 256 * 256
    assert torch.equal(got.data[planes:planes + want.numel()].view_as(want), want)


# (Nb, C, H, O, k), pool, (I, F), whether the pooling runs in the launch: rectangles of one to eight tiles, with whole and half
# limits, beside layers whose single launch would leave waves idle
POOL_ROUTES = [((1, 128, 14, 128, 3), (2, 2, 0), (16, 16), False), ((3, 256, 13, 256, 3), (3, 2, 0), (16, 16), False), ((128, 64, 16, 128, 3), (2, 2, 0), (16, 16), True),
               ((40, 16, 28, 40, 3), (2, 2, 0), (16, 16), True), ((33, 64, 13, 96, 1), (3, 2, 1), (16, 16), True), ((70, 64, 8, 70, 3), (2, 2, 0), (3, 5), True),
               ((9, 512, 6, 512, 3), (2, 2, 0), (3, 5), False), ((5, 20, 31, 64, 5), (5, 1, 2), (3, 5), True)]


@pytest.mark.parametrize("shape,pool,act,fused", POOL_ROUTES, ids=lambda v: str(v).replace(" ", ""))
def test_pooled_layers_agree_on_both_routes(monkeypatch, shape, pool, act, fused):
    """A pooled layer as modules route it -- in one launch, which hands operands on, or as sums and a pass of its own -- against
    the separate pass."""
    Nb, C, H, O, k = shape
    torch.manual_seed(3)
    layer = modules.Conv2dShift(C, O, k, padding=k // 2, use_kernel=True, act_integer_bits=act[0], act_fraction_bits=act[1]).to(DEV).eval()
    layer.shift.data = torch.randint(-14, 1, layer.shift.shape, device=DEV).float()
    layer.shift.data.view(-1)[0] = -14
    layer.sign.data = torch.randint(0, 2, layer.sign.shape, device=DEV).float() * 2 - 1
    x = torch.randn(Nb, C, H, H, device=DEV) * (40 if act[0] == 16 else 1)
    scale, shift = torch.randn(O, device=DEV) * 0.1, torch.randn(O, device=DEV)
    emit = ((1, 1), *act, True, torch.int8 if act[0] + act[1] <= 8 else torch.int32)
    with torch.no_grad():
        def run():
            return modules.conv_kernel_forward(layer, x, layer.packed_weights(), scale, shift, None, True, False, emit, pool,
                                               emit_filter=(3, 3))

        f, q = run()
        assert isinstance(q, kernels.Prepared) == fused
        monkeypatch.setattr(modules, "_FUSE_EPILOGUE", False)
        want_f, want_q = run()
    assert torch.equal(f, want_f) and torch.equal(q.padded() if fused else q, want_q)


@pytest.mark.parametrize("x_bytes", [4, 1])
def test_the_long_signatures_answer_like_the_packed_one(rng, x_bytes):
    """ds_mfma_conv2d (sums; float, padded and operand results, from a window of the prepared tensor) and ds_mfma_conv2d_pool, as a
    caller of the library writes them, against the arrays that the package sends."""
    lib = kernels._lib
    Nb, C, H, W, O, top = 2, 40, 13, 11, 70, 6
    F_in, I, F, dtype = (16, 16, 16, torch.int32) if x_bytes == 4 else (5, 3, 5, torch.int8)
    stream = lib.stream_handle(torch.device(DEV))
    _, _, cw = _weights(rng, (O, C, 2, 3), top, ternary=True)
    _, _, inner = _weights(rng, (O, C, 1, 2), top, ternary=True)
    bias = _dev(rng.integers(-2 ** 20, 2 ** 20, size=O).astype(np.int32))
    scale, shift = torch.randn(O, device=DEV), torch.randn(O, device=DEV)
    prepared, blob, at = kernels.mfma_route(_dev(_activations(rng, (Nb, C, H, W), x_bytes, 1 << 22)), (1, 2), cw, O, (2, 3), x_bytes)
    inner_blob = kernels._mfma_of(inner, at, x_bytes, O, C, 1, 2)
    sizes = (Nb, C, H + 2, W + 4, O)
    OH, OW = (H + 2 - 2) // 2 + 1, W + 4 - 3 + 1
    y = torch.empty(Nb, O, OH, OW, dtype=torch.int32, device=DEV)
    lib.call("ds_mfma_conv2d", lib.ptr(prepared.data), lib.ptr(blob), lib.ptr(bias), lib.ptr(y), None, None, None, None, None, *sizes,
             2, 3, 2, 1, 0, 0, 2, 3, 0, at, x_bytes, 0, 0, 16, 16, 0, 0, 4, 1, 1, 0, 0, 0, stream)
    assert torch.equal(y, kernels.mfma_conv2d(prepared, blob, bias, O, (2, 3), (2, 1), at))
    # the centre of the prepared tensor, read by a filter of one row
    residual = torch.randn(Nb, O, H, (W - 2) // 2 + 1, device=DEV)
    args = (prepared, inner_blob, bias, O, (1, 2), (1, 2), at, (1, 2), F_in, scale, shift, residual, True)
    for filt in (None, (3, 3)):
        want_f, want_q = kernels.mfma_conv2d(*args, ((2, 1), I, F, dtype, filt))
        out, q = torch.empty_like(want_f), torch.empty_like(want_q if filt is None else want_q.data)
        lib.call("ds_mfma_conv2d", lib.ptr(prepared.data), lib.ptr(inner_blob), lib.ptr(bias), None, lib.ptr(out), lib.ptr(q),
                 lib.ptr(scale), lib.ptr(shift), lib.ptr(residual), *sizes, 1, 2, 1, 2, 1, 2, 2, 3, 0, at, x_bytes, F_in, 1, I, F, 2, 1,
                 x_bytes | (0 if filt is None else lib.DS_Q_OPERANDS), *(filt or (1, 1)), 0, 0, 0, stream)
        got = q if filt is None else kernels.Prepared(q, want_q.dims, filt, 0, x_bytes, (2, 1)).padded()
        assert torch.equal(out, want_f) and torch.equal(got, want_q if filt is None else want_q.padded())
    # operands from a convolution's epilogue, and a max pooling behind the layer that reads them
    _, _, cw2 = _weights(rng, (64, O, 3, 3), top, ternary=True)
    blob2, bias2 = kernels._mfma_of(cw2, at, x_bytes, 64, O, 3, 3), _dev(rng.integers(-2 ** 20, 2 ** 20, size=64).astype(np.int32))
    scale2, shift2 = torch.randn(64, device=DEV), torch.randn(64, device=DEV)
    args = (want_q, blob2, bias2, 64, (3, 3), (1, 1), at, 0, F_in, scale2, shift2, None, True)
    for filt in (None, (3, 3)):
        pooled_f, pooled_q = kernels.mfma_conv2d(*args, ((1, 2), I, F, dtype, filt), True, None, (3, 2, 1))
        out, q = torch.empty_like(pooled_f), torch.empty_like(pooled_q if filt is None else pooled_q.data)
        lib.call("ds_mfma_conv2d_pool", lib.ptr(want_q.data), lib.ptr(blob2), lib.ptr(bias2), lib.ptr(out), lib.ptr(q), lib.ptr(scale2),
                 lib.ptr(shift2), *want_q.dims, 64, 3, 3, 1, 1, 3, 3, at, x_bytes, F_in, 1, I, F, 1, 2,
                 x_bytes | (0 if filt is None else lib.DS_Q_OPERANDS), *(filt or (1, 1)), 1, 2, 1, 3, 2, 1, stream)
        got = q if filt is None else kernels.Prepared(q, pooled_q.dims, filt, 0, x_bytes, (1, 2)).padded()
        assert torch.equal(out, pooled_f) and torch.equal(got, pooled_q if filt is None else pooled_q.padded())


def test_windows_without_a_form_keep_their_pass():
    serves = kernels._lib.lib().ds_mfma_pool_serves
    assert serves(8, 8, 3, 2, 1) == 1 and serves(1, 1, 1, 1, 0) == 1 and serves(11, 11, 11, 1, 0) == 1
    assert serves(8, 8, 12, 1, 0) == 0 and serves(8, 8, 3, 2, 2) == 0 and serves(2, 8, 3, 1, 0) == 0 and serves(8, 8, 3, 0, 1) == 0
    assert not kernels.mfma_pool_serves(1, 8, 8, 32, (3, 2, 1)) and not kernels.mfma_pool_serves(64, 1024, 1024, 64, (3, 2, 1))


@pytest.mark.parametrize("x_bytes", [4, 1])
@pytest.mark.parametrize("O", [64, 40])
def test_scales_without_a_shorter_epilogue(rng, x_bytes, O):
    """Constants that powers of two cannot be multiplied into -- a scale next to the smallest floats, one whose product with
    2^-F has no normal form, huge and infinite ones, NaN -- beside ordinary ones, in launches with many tiles, whose epilogue
    multiplies them in where it can: float and quantised results against the separate pass."""
    C, Nb, H, k = 32, 33, 33, 1
    F_in, I, F, dtype = (16, 16, 16, torch.int32) if x_bytes == 4 else (5, 3, 5, torch.int8)
    s, sign, cw = _weights(rng, (O, C, k, k), 6, ternary=False)
    x = _dev(_activations(rng, (Nb, C, H, H), x_bytes, 1 << 18))
    prepared, blob, top = kernels.mfma_route(x, 0, cw, O, (k, k), x_bytes)
    y = kernels.mfma_conv2d(prepared, blob, None, O, (k, k), 1, top)
    for at, scale_at, shift_at in ((None, None, None), (3, 2.0 ** -120 * 1.2345678, 0.5), (5, 1.1e-38, 0.0), (7, 1e-45, 1e-45),
                                   (9, float("inf"), 0.0), (1, float("nan"), 1.0), (2, 3e38, -3e38), (0, 0.0, float("nan")),
                                   (4, -2.0 ** 70, 2.0 ** 70), (6, 1.0, float("inf"))):
        scale, shift = torch.rand(O, device=DEV) + 0.5, torch.randn(O, device=DEV)
        if at is not None:
            scale[at], shift[at] = scale_at, shift_at
        for relu in (True, False):
            f, q = kernels.requantize_affine_pad(y, F_in, scale, shift, None, relu, (1, 1), I, F, True, dtype)
            args = (prepared, blob, None, O, (k, k), 1, top, 0, F_in, scale, shift, None, relu, ((1, 1), I, F, dtype))
            out, got = kernels.mfma_conv2d(*args, True)
            assert torch.equal(out.view(torch.int32), f.view(torch.int32)) or torch.equal(torch.nan_to_num(out, nan=7.0),
                                                                                        torch.nan_to_num(f, nan=7.0))
            assert torch.equal(got, q)
            assert torch.equal(kernels.mfma_conv2d(*args, False)[1], q)


# (tiles of 64 channels x 32 pixels per CU at least, x_bytes, C, O, images of H x W): launches whose whole tiles end with
# workgroups on some CUs only, by how much is left and how long the reduction is; the last tiles end inside one
UNEVEN = [(4, 4, 32, 64, (5, 91, 91)), (4, 1, 40, 70, (3, 85, 83)), (5, 4, 70, 128, (6, 61, 61)), (6, 1, 128, 256, (49, 15, 17)),
          (6, 4, 128, 100, (7, 59, 60)), (4, 4, 320, 640, (1, 61, 71))]


@pytest.mark.parametrize("x_bytes,C,O,images", [c[1:] for c in UNEVEN], ids=lambda v: str(v).replace(" ", ""))
def test_tiles_that_are_left_are_shared(oracle, rng, x_bytes, C, O, images):
    """Sums against the oracle, and the epilogue of whole and shared tiles against the separate pass, with digits 3 and 4 in
    the shared ones."""
    Nb, H, W = images
    tiles = -(-Nb * H * W // 32) * -(-O // 64)
    assert tiles > 1024
    s, sign, cw = _weights(rng, (O, C, 3, 3), 14, ternary=False)
    x = _activations(rng, (Nb, C, H, W), x_bytes, 1 << 18)
    if x_bytes == 4:
        x[-1, :, -2:] <<= 6
        x[-1, ..., -1] = -2 ** 31
    bias = rng.integers(-2 ** 20, 2 ** 20, size=O).astype(np.int32)
    prepared, blob, top = kernels.mfma_route(_dev(x), 1, cw, O, (3, 3), x_bytes)
    y = kernels.mfma_conv2d(prepared, blob, _dev(bias), O, (3, 3), 1, top)
    xp = np.pad(x.astype(np.int32), ((0, 0), (0, 0), (1, 1), (1, 1)))
    np.testing.assert_array_equal(y.cpu().numpy(), oracle.conv2d(xp, -s.astype(np.int32), sign.astype(np.int32), bias, (1, 1),
                                                                 nthreads=16))
    F_in, I, F, dtype = (16, 16, 16, torch.int32) if x_bytes == 4 else (5, 3, 5, torch.int8)
    scale, shift, res = (torch.rand(O, device=DEV) + 0.5), torch.randn(O, device=DEV), torch.randn(y.shape, device=DEV)
    f, q = kernels.requantize_affine_pad(y, F_in, scale, shift, res, True, (1, 1), I, F, True, dtype)
    args = (prepared, blob, _dev(bias), O, (3, 3), 1, top, 0, F_in, scale, shift, res, True, ((1, 1), I, F, dtype, (3, 3)))
    out, handed = kernels.mfma_conv2d(*args, True)
    assert torch.equal(out, f) and torch.equal(handed.padded(), q)

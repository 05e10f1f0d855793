"""GPU: the buffers that fused layers hand to each other, where a model runs on several streams, is captured into a graph,
or is called with other sizes in between."""
import pytest
import torch
import torch.nn as nn

from deepshift_amd import _lib, convert, fuse, kernels, modules
from tests.conftest import Tune

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
FORMATS = [(16, 16), (3, 5)]


def _model(I, F, seed=0, widths=((32, 64, 3), (64, 64, 1), (64, 64, 3), (64, 32, 1)), weight_bits=5, scale=None):
    """Fused convolutions with padded and unpadded hand-offs."""
    torch.manual_seed(seed)
    layers = []
    for C, O, k in widths:
        layers += [nn.Conv2d(C, O, k, padding=k // 2, bias=False), nn.BatchNorm2d(O), nn.ReLU()]
        if scale:                                      # no weight below 2^-14
            nn.init.uniform_(layers[-3].weight, scale / 100, scale)
    model, n = convert.convert_to_shift(nn.Sequential(*layers).eval(), 1000, "PS", convert_weights=True, use_kernel=True,
                                        weight_bits=weight_bits, act_integer_bits=I, act_fraction_bits=F)
    assert n == len(widths)
    return fuse.fuse_conv_epilogues(model.to(DEV))


def _inputs(n, Nb=16, C=32, H=56):
    g = torch.Generator(device=DEV).manual_seed(Nb)
    return [torch.rand(Nb, C, H, H, generator=g, device=DEV) * 2 for _ in range(n)]


@pytest.mark.parametrize("I,F", FORMATS)
def test_two_streams_share_a_model(I, F):
    """Passes of two streams alternate with nothing between them but the host."""
    with torch.no_grad():
        model = _model(I, F)
        xs = _inputs(12)
        want = [model(x) for x in xs]
        torch.cuda.synchronize()
        streams = [torch.cuda.Stream(), torch.cuda.Stream()]
        got = []
        for i, x in enumerate(xs):
            with torch.cuda.stream(streams[i % 2]):
                got.append(model(x))
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("I,F", FORMATS)
def test_a_captured_pass_owns_its_buffers(I, F):
    """Eager passes right after a capture (which executes nothing), replays, and eager passes of another size between
    the replays: each result is that of a pass by itself."""
    with torch.no_grad():
        model = _model(I, F)
        small, large = _inputs(4, 2, H=15), _inputs(4, 5, H=15)
        want_small, want_large = [model(x) for x in small], [model(x) for x in large]
        model(_inputs(1, 3, H=9)[0])       # what is kept now fits neither
        static = small[0].clone()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = model(static)
        assert torch.equal(model(small[1]), want_small[1])
        for i in range(4):
            static.copy_(small[i])
            graph.replay()
            assert torch.equal(model(large[i]), want_large[i])
            assert torch.equal(y, want_small[i])
            graph.replay()
            assert torch.equal(model(small[3 - i]), want_small[3 - i])
            assert torch.equal(y, want_small[i])


def _chain(widths):
    torch.manual_seed(1)
    layers = []
    for K, N in zip(widths[:-1], widths[1:]):
        layers += [nn.Linear(K, N), nn.ReLU()]
    model, _ = convert.convert_to_shift(nn.Sequential(*layers[:-1]).eval(), 0, "PS", convert_weights=True, use_kernel=True)
    fused = fuse.fuse_conv_epilogues(model.to(DEV))
    assert any(isinstance(m, fuse.FusedLinearChain) for m in fused.modules())
    return fused


@pytest.mark.parametrize("widths", [(64, 64, 32, 8), (784, 512, 512, 10)], ids=["one launch", "launch per layer"])
def test_streams_and_graphs_have_their_own_chain_workspace(widths):
    with torch.no_grad():
        model = _chain(widths)
        chain = next(m for m in model.modules() if isinstance(m, fuse.FusedLinearChain))
        g = torch.Generator(device=DEV).manual_seed(2)
        xs = [torch.rand(64, widths[0], generator=g, device=DEV) for _ in range(16)]
        want = [model(x) for x in xs]
        torch.cuda.synchronize()
        streams, got = [torch.cuda.Stream(), torch.cuda.Stream()], []
        for i, x in enumerate(xs):
            with torch.cuda.stream(streams[i % 2]):
                got.append(model(x))
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        static = xs[0].clone()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = model(static)
        assert chain.status() == 0 and torch.equal(model(xs[1]), want[1])
        for i in range(4):
            static.copy_(xs[i])
            graph.replay()
            assert torch.equal(model(xs[i + 4][:30]), want[i + 4][:30])
            assert torch.equal(y, want[i])
        assert chain.status() == 0


def test_replays_report_a_barrier_that_gave_up():
    """The test hook makes the barriers of a captured launch wait, 200 us at most, for one arrival more than the grid has."""
    with torch.no_grad():
        model = _chain((64, 64, 32, 8))
        chain = next(m for m in model.modules() if isinstance(m, fuse.FusedLinearChain))
        x = torch.rand(64, 64, device=DEV)
        want = model(x)
        torch.cuda.synchronize()
        graphs = []
        for knobs in (dict(), dict(chain_spin_us=200, chain_extra=1)):
            graphs.append(torch.cuda.CUDAGraph())
            with Tune(**knobs), torch.cuda.graph(graphs[-1]):
                y = model(x)
            if not knobs:
                first = y
        graphs[0].replay()
        assert chain.status() == 0 and torch.equal(first, want)
        graphs[1].replay()
        assert chain.status() == 1
        graphs[0].replay()
        assert chain.status() == 1 and torch.equal(first, want) and torch.equal(model(x), want)


@pytest.mark.parametrize("M", [1024, 64])
def test_what_a_capture_builds_is_not_kept(M):
    """A capture records the layout passes of weights and bias and runs none of them: an eager call between capture and
    first replay builds its own.  1024 rows take another kernel than the rows that warmed the layer up."""
    torch.manual_seed(3)
    layer = modules.LinearShift(512, 512, use_kernel=True).to(DEV)
    layer.sign.data.copy_(torch.randint(0, 2, layer.sign.shape).float() * 2 - 1)
    x = torch.randn(M, 512, device=DEV)
    junk = torch.full((64 << 20,), 0x55, dtype=torch.uint8, device=DEV)
    del junk                              # what is allocated next holds something
    with torch.no_grad():
        if M > 64:
            want = torch.cat([layer(x[i:i + 64]) for i in range(0, M, 64)])
        else:
            layer.packed_weights()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = layer(x)
        got = layer(x)
        if M == 64:
            graph_reads = layer.conc_weight
            layer.conc_weight = None      # start over
            layer._fixed_bias = modules._FixedBias()
            want = layer(x)
        assert torch.equal(got, want)
        for _ in range(3):
            y.zero_()
            graph.replay()
            assert torch.equal(layer(x), want)
            assert torch.equal(y, want)
        assert M > 64 or graph_reads.data is not layer.conc_weight.data


@pytest.mark.parametrize("changed", [[1], [2], [1, 2, 3]], ids=str)
def test_weights_loaded_after_fusing_may_need_the_older_kernels(changed):
    """Shifts past 14 in layers that were fused for the operand layout: the layer before hands it over, the layer reads
    it back."""
    with torch.no_grad():
        model = _model(16, 16, weight_bits=6, scale=0.3)
        convs = [m for m in model.modules() if isinstance(m, modules.Conv2dShift)]
        x = _inputs(1, 3, H=11)[0]
        assert all(int(c.packed_weights().max_field) <= 14 for c in convs)
        model(x)
        for i in changed:
            convs[i].shift.view(-1)[::7] = -15.0 - (i % 2) * 5
        got = model(x)
        assert all((int(c.packed_weights().max_field) > 14) == (i in changed) for i, c in enumerate(convs))
        bns = [m for m in model.modules() if isinstance(m, fuse.FusedConv2dShift)]
        want = x
        for fused in bns:
            y = kernels.conv2d(kernels.quantize(want), fused.conv.shift, fused.conv.sign, None, fused.conv.packed_weights(),
                               1, fused.conv.padding)
            want = kernels.dequantize_affine(y, 16, fused.scale, fused.shift, None, True)
        assert torch.equal(got, want)


def test_a_pair_whose_weights_reach_shift_15(rng):
    """Both convolutions of a down-sampling block: the one-launch pair on the padded tensor serves them."""
    from deepshift_amd import workloads
    g = torch.Generator().manual_seed(7)
    model = workloads.randomize_batchnorm(workloads.ResNet18(), g).eval()
    model, _ = convert.convert_to_shift(model, 1000, "PS", convert_weights=True, use_kernel=True, weight_bits=6)
    model = model.to(DEV)
    x = torch.randn(2, 3, 64, 64, generator=g).to(DEV)
    with torch.no_grad():
        for m in model.modules():
            if isinstance(m, modules.Conv2dShift):
                m.shift.clamp_(-14, 0)
        fused = fuse.fuse_conv_epilogues(model)
        pair = next(m for m in fused.modules() if isinstance(m, fuse.FusedShortcutPair))
        fused(x)
        for conv in (pair.first.conv, pair.shortcut.conv):
            conv.shift.view(-1)[:100] = -15.0
        got = fused(x)
        assert all(f.conv.packed_weights().max_field == 15 for f in (pair.first, pair.shortcut))
        assert torch.equal(got, fuse.fuse_conv_epilogues(model, handoff=False)(x))


@pytest.mark.parametrize("x_bytes,O", [(4, 40), (4, 12), (1, 33), (1, 64)])
@pytest.mark.parametrize("pad", [(1, 1), (2, 0), (0, 3), (0, 0)])
def test_a_buffer_that_nobody_zeroed_gets_its_border(x_bytes, O, pad):
    """The operand layout written into memory full of other values: border and unused channels included, it holds what
    the padded tensor does."""
    from tests.test_gpu_mfma import _activations, _weights
    import numpy as np
    rng = np.random.default_rng(O)
    dtype, I, F = (torch.int32, 16, 16) if x_bytes == 4 else (torch.int8, 3, 5)
    s, sign, cw = _weights(rng, (O, 24, 3, 3), 14, ternary=False)
    x = torch.from_numpy(_activations(rng, (3, 24, 11, 9), x_bytes, 1 << 20)).to(DEV)
    prepared, blob, top = kernels.mfma_route(x, (1, 1), cw, O, (3, 3), x_bytes)
    args = (prepared, blob, None, O, (3, 3), (1, 1), top, 0, F, None, None, None, False)
    _, want = kernels.mfma_conv2d(*args, (pad, I, F, dtype), False)
    junk = torch.full((1 << 22,), 0x55, dtype=torch.uint8, device=DEV)
    del junk                                # the allocator's next blocks hold 0x55
    _, got = kernels.mfma_conv2d(*args, (pad, I, F, dtype, (3, 3)), False)
    assert torch.equal(got.padded(), want)
    _, _, cw2 = _weights(rng, (48, O, 3, 3), 14, ternary=False)
    blob2 = kernels._mfma_of(cw2, 14, x_bytes, 48, O, 3, 3)
    y = kernels.mfma_conv2d(got, blob2, None, 48, (3, 3), (1, 1), 14)
    again = kernels.mfma_conv2d(kernels.mfma_prepare(want, 0, (3, 3), x_bytes), blob2, None, 48, (3, 3), (1, 1), 14)
    assert torch.equal(y, again)


@pytest.mark.parametrize("fmt", [(0, 16), (20, 20), (12, -4), (1, 5)], ids=str)
def test_modules_refuse_what_their_conversion_refuses(fmt):
    """Formats past 32 bits or without an integer bit (1.5 is the reference's one-bit format: served), inputs on the host or
    without a batch."""
    I, F = fmt
    conv = modules.Conv2dShift(64, 64, 3, padding=1, bias=False, use_kernel=True, act_integer_bits=I, act_fraction_bits=F).to(DEV)
    linear = modules.LinearShift(2112, 64, bias=False, use_kernel=True, act_integer_bits=I, act_fraction_bits=F).to(DEV)
    with torch.no_grad():
        for layer, x in ((conv, torch.zeros(1, 64, 8, 8, device=DEV)), (linear, torch.zeros(3, 2112, device=DEV))):
            if I == 1:
                assert layer(x).device.type == "cuda"
                with pytest.raises(TypeError):
                    layer(x.cpu())
            else:
                with pytest.raises(_lib.DeepShiftError):
                    layer(x)
        if I == 1:
            with pytest.raises(TypeError):
                conv(torch.zeros(64, 8, 8, device=DEV))


@pytest.mark.parametrize("C,O,top", [(24, 40, 14), (8, 8, 14), (24, 40, 20)])
@pytest.mark.parametrize("pad", [(1, 1), (2, 1), (3, 2)])
def test_circular_padding_is_made_once(monkeypatch, C, O, top, pad):
    """... on whichever kernel the layer runs: matrix cores, few channels, shifts past 14."""
    torch.manual_seed(4)
    layer = modules.Conv2dShift(C, O, 3, padding=pad, padding_mode="circular", use_kernel=True, weight_bits=6, bias=False).to(DEV)
    layer.shift.data.copy_(torch.randint(-top, 1, layer.shift.shape).float())
    layer.shift.data.view(-1)[0] = -top
    layer.sign.data.copy_(torch.randint(0, 2, layer.sign.shape).float() * 2 - 1)
    x = torch.randn(2, C, 9, 7, device=DEV)
    made = []
    real = modules._circular_pad
    monkeypatch.setattr(modules, "_circular_pad", lambda *a: made.append(1) or real(*a))
    with torch.no_grad():
        got = layer(x)
        assert len(made) == 1
        y = kernels.conv2d(kernels.quantize(real(x, pad)), layer.shift, layer.sign, None, layer.packed_weights())
        assert torch.equal(got, kernels.dequantize(y))


def test_forward_hooks_read_a_hand_off_as_a_tensor():
    import copy
    with torch.no_grad():
        model = _model(16, 16)
        x = _inputs(1, 2, H=9)[0]
        seen = []

        def hook(module, args, out):
            if isinstance(out, kernels.Prepared):
                seen.append((tuple(out.shape), out.dtype, out.device, out.dim(), out.size(1), out.float().mean().item(),
                             int(torch.count_nonzero(out)), torch.equal(out, out.padded()), tuple(out[0, :2].shape)))

        for m in model.modules():
            if isinstance(m, fuse.FusedConv2dShift):
                m.register_forward_hook(hook)
        want = model(x)
        assert len(seen) == 3
        for shape, dtype, device, dim, channels, mean, count, same, first in seen:
            assert len(shape) == dim == 4 and channels == shape[1] == 64 and dtype == torch.int32 and device == x.device
            assert mean > 0 and count > 0 and same and first == (2,) + shape[2:]
        q = model.get_submodule("fused_0")(x)
        assert not hasattr(q, "no_such_name") and copy.copy(q).dims == q.dims
        assert torch.equal(model(x), want)


@pytest.mark.parametrize("C,O,k,Nb,H,matrix", [(4, 64, 1, 2, 9, False), (31, 128, 1, 40, 30, False), (32, 127, 1, 40, 30, False),
                                               (32, 128, 1, 2, 9, False), (32, 128, 1, 40, 30, True), (40, 17, 1, 2, 9, False), (41, 17, 1, 2, 9, True),
                                               (64, 16, 1, 270, 32, False), (64, 17, 1, 270, 32, True), (64, 16, 1, 2, 9, True),
                                               (4, 140, 3, 40, 30, False), (5, 40, 3, 2, 11, True)])
def test_unpadded_integer_convolutions_take_the_kernel_that_pays(oracle, monkeypatch, C, O, k, Nb, H, matrix):
    """kernels.conv2d on both sides of every line of its rule, against the oracle; padded inputs are not asked."""
    from tests.test_gpu_mfma import _activations, _weights
    import numpy as np
    rng = np.random.default_rng(C * O)
    s, sign, cw = _weights(rng, (O, C, k, k), 14, ternary=False)
    x = _activations(rng, (Nb, C, H, H), 4, 1 << 24)
    launches = []
    real = kernels.mfma_conv2d
    monkeypatch.setattr(kernels, "mfma_conv2d", lambda *a, **kw: launches.append(1) or real(*a, **kw))
    args = [torch.from_numpy(np.ascontiguousarray(a)).to(DEV) for a in (x, -s.astype(np.int32), sign.astype(np.int32))]
    got = kernels.conv2d(*args, None, cw)
    assert len(launches) == matrix
    want = oracle.conv2d(x, -s.astype(np.int32), sign.astype(np.int32), None, (1, 1), nthreads=16)
    np.testing.assert_array_equal(got.cpu().numpy(), want)
    padded = kernels.conv2d(*args, None, cw, 1, 1)
    assert len(launches) == matrix + 1
    assert k > 1 or torch.equal(padded[:, :, 1:-1, 1:-1], got)


@pytest.mark.parametrize("M,widths,alone", [(64, (784, 512, 512, 10), False), (512, (784, 1024, 1024, 10), True),
                                            (4, (3072, 64, 8), False)])
def test_chains_and_single_layers_follow_one_rule(monkeypatch, M, widths, alone):
    """A chain is one call of the library while its layers are small; large ones take the matrix cores there as they do
    alone."""
    calls = []
    real = kernels.linear_chain
    monkeypatch.setattr(kernels, "linear_chain", lambda *a: calls.append(1) or real(*a))
    with torch.no_grad():
        model = _chain(widths)
        x = torch.rand(M, widths[0], device=DEV)
        got = model(x)
        assert bool(calls) != alone
        chain = next(m for m in model.modules() if isinstance(m, fuse.FusedLinearChain))
        want = x
        for layer, relu in zip(chain.linears, chain.relus):
            want = torch.relu(layer(want)) if relu else layer(want)
        assert torch.equal(got, want)

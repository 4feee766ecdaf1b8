"""3x3 convolutions against packed weights (fluidml_hip_conv3x3_packed_chain) on the GPU, at the edges of its tiles,
channel chunks, filter groups and splits, against the oracle; and the values its bf16 parts cannot carry."""
import ctypes
import os

import numpy as np
import pytest

from oracle import graph_runner
from oracle import kernels as ok
from tests.util import DeviceView, assert_close, some_layouts

pytestmark = pytest.mark.gpu
RELU = [("EW_RELU", 0.0)]


def _run(device, x, w, bias, pads, parts, tile=0, splits=0, chain=RELU, layouts=(None, None, None), times=1):
    import torch

    from fluidml_amd import cabi

    N, _, H, W = x.shape
    F = w.shape[0]
    shape = (N, F, H + pads[0] + pads[2] - 2, W + pads[1] + pads[3] - 2)
    dx, dw = DeviceView(ok.View(x, layouts[0]), device), DeviceView(ok.View(w, layouts[1]), device)
    db = DeviceView(ok.View(bias), device) if bias is not None else None
    do = DeviceView(ok.View.empty(shape, layout=layouts[2], fill=9), device)
    size = ctypes.c_size_t()
    cabi.call("conv3x3_packed_bytes", dw.ref(), parts, ctypes.byref(size))
    packed = torch.zeros(size.value, dtype=torch.uint8, device=device)
    cabi.call("conv3x3_pack", dw.ref(), parts, packed.data_ptr(), None)
    program = cabi.make_chain([(getattr(cabi, op), c) for op, c in chain])
    for _ in range(times):  # (again: the arrival counters of a split launch are back at zero)
        cabi.call("conv3x3_packed_chain", dx.ref(), dw.ref(), packed.data_ptr(), parts, db.ref() if db else None, do.ref(),
                  cabi.i64_array(pads), ctypes.byref(program), tile << 4 | splits << 8, None)
    return do.logical()


def _oracle(x, w, bias, pads, relu=True):
    N, _, H, W = x.shape
    out = ok.View.empty((N, w.shape[0], H + pads[0] + pads[2] - 2, W + pads[1] + pads[3] - 2))
    ok.conv(ok.View(x), ok.View(w), ok.View(bias) if bias is not None else None, out, pads, [1, 1], [1, 1], 1)
    return np.maximum(out.logical(), 0) if relu else out.logical()


def _operands(seed, N, C, H, W, F):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((N, C, H, W), np.float32), (rng.standard_normal((F, C, 3, 3)) * (C * 9) ** -0.5).astype(np.float32),
            rng.standard_normal(F).astype(np.float32))


@pytest.mark.parametrize("N,C,H,W,F,pads", [
    (1, 16, 8, 16, 128, [1, 1, 1, 1]),    # one workgroup of four filter tiles
    (1, 16, 16, 16, 64, [1, 1, 1, 1]),    # two filter tiles, two rows of waves
    (2, 32, 9, 17, 65, [1, 1, 1, 1]),     # one past every tile
    (1, 48, 7, 15, 127, [1, 1, 1, 1]),    # one short of it
    (1, 17, 10, 20, 32, [0, 0, 0, 0]),    # channels and pads that leave remainders
    (1, 5, 3, 3, 33, [0, 0, 0, 0]),       # a single output pixel
    (3, 31, 5, 33, 96, [2, 0, 1, 2]),
    (1, 160, 6, 6, 160, [1, 1, 1, 1]),    # split by the library's rule
])
@pytest.mark.parametrize("tile,splits", [(0, 0), (1, 1), (2, 1), (1, 3), (2, 2)])
def test_packed_conv(device, N, C, H, W, F, pads, tile, splits):
    x, w, bias = _operands(7, N, C, H, W, F)
    print("[case]", N, C, H, W, F, pads, tile, splits, flush=True)
    got = _run(device, x, w, bias, pads, 3, tile, splits, times=3)
    assert_close(got, _oracle(x, w, bias, pads), what="three parts")
    def rounded(v):  # to bf16, nearest even
        bits = v.view(np.uint32).astype(np.uint64)
        return ((bits + 0x7FFF + ((bits >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)
    got = _run(device, x, w, None, pads, 1, tile, splits, chain=[])
    assert_close(got, _oracle(rounded(x), rounded(w), None, pads, relu=False), what="bf16")


@pytest.mark.parametrize("N,C,H,W,F,tile", [
    (1, 16, 10, 18, 64, 1),      # a single chunk
    (1, 17, 10, 18, 128, 2),     # two, the second of one channel
    (2, 48, 9, 20, 160, 1),      # three: the second set of registers stays behind
    (1, 80, 12, 7, 96, 2),       # five
    (8, 40, 140, 60, 64, 1),     # more than two workgroups per compute unit: 576 of 64 filters, the last chunk half full
    (3, 16, 171, 62, 130, 1),    # 1032 of 128 filters, half of them nearly empty
])
def test_packed_conv_bf16_chunks(device, N, C, H, W, F, tile):
    """Exact: operands of a few bits, so that every product and every sum of them is a float32."""
    print("[case]", N, C, H, W, F, tile, flush=True)
    rng = np.random.default_rng(5)
    x = rng.integers(-8, 9, (N, C, H, W)).astype(np.float32)
    w = rng.integers(-4, 5, (F, C, 3, 3)).astype(np.float32)
    bias = rng.integers(-16, 17, F).astype(np.float32)
    got = _run(device, x, w, bias, [1, 1, 1, 1], 1, tile, 1)
    np.testing.assert_array_equal(got, _oracle(x, w, bias, [1, 1, 1, 1]))


def _recorded(device, N, C, H, W, F, parts, tile=0, splits=0, pool=False):
    """What a convolution launches: (kernel's name, workgroups a compute unit holds, grid, bytes of scratch)."""
    import torch

    from fluidml_amd import cabi
    from util import launched

    shape = (N, F, H // 2, W // 2) if pool else (N, F, H, W)
    x, w, b, out = (torch.zeros(*s, device=device) for s in ((N, C, H, W), (F, C, 3, 3), (F,), shape))
    ref = lambda t: ctypes.byref(cabi.make_tensor(t.data_ptr(), cabi.FL_FLOAT32, t.shape, t.stride()))
    size = ctypes.c_size_t()
    cabi.call("conv3x3_packed_bytes", ref(w), parts, ctypes.byref(size))
    packed = torch.zeros(size.value, dtype=torch.uint8, device=device)
    name = "conv3x3_packed_chain_pool" if pool else "conv3x3_packed_chain"
    call = lambda s: cabi.call(name, ref(x), ref(w), packed.data_ptr(), parts, ref(b), ref(out), cabi.i64_array([1] * 4),
                               ctypes.byref(cabi.make_chain([])), tile << 4 | splits << 8, s)
    found, = launched(call, first_on_its_stream=True)
    assert "ConvPartsKernel" in found[0]
    return found


@pytest.mark.parametrize("C", [64, 40])
@pytest.mark.parametrize("F,tile", [(128, 1), (128, 2), (64, 1), (64, 2)])
@pytest.mark.parametrize("pool", [False, True])
def test_packed_conv_bf16_of_many_workgroups_fits(device, C, F, tile, pool):
    """No launch of more than two workgroups per compute unit has splits, and none holds registers for their exchange."""
    name, fit, grid, scratch = _recorded(device, 8, C, 160, 112, F, 1, tile, 1, pool)
    assert grid[0] > 512 and fit >= 3 and scratch == 0, (name, fit, grid, scratch)


@pytest.mark.parametrize("C", [16, 64, 65, 80, 256, 320])
@pytest.mark.parametrize("F,tile,splits", [(128, 1, 1), (64, 2, 1), (96, 1, 4), (48, 2, 4), (96, 2, 8)])
@pytest.mark.parametrize("pool", [False, True])
def test_packed_conv_bf16_chunks_ahead(device, C, F, tile, splits, pool):
    """Two chunks of activations are in flight where a workgroup has five and more, four of split channels; the sums are the same either way.  Exact:
    operands of a few bits, so that every product and every sum of them is a float32."""
    print("[case]", C, F, tile, splits, pool, flush=True)
    chunks = -(-C // 16)
    per = -(-chunks // splits)
    name, _, grid, _ = _recorded(device, 2, C, 20, 35, F, 1, tile, splits, pool)
    assert f"ELi{2 if per >= (4 if per < chunks else 5) else 1}ELb1EE" in name, (name, grid, per)
    if pool:
        return
    rng = np.random.default_rng(C + F)
    x = rng.integers(-8, 9, (2, C, 20, 35)).astype(np.float32)
    w = rng.integers(-4, 5, (F, C, 3, 3)).astype(np.float32)
    bias = rng.integers(-16, 17, F).astype(np.float32)
    got = _run(device, x, w, bias, [1, 1, 1, 1], 1, tile, splits, times=2)
    np.testing.assert_array_equal(got, _oracle(x, w, bias, [1, 1, 1, 1]))


@pytest.mark.parametrize("N,C,hw,F,workgroups", [
    # three parts, two tiles per wave; the partial tiles of few workgroups are cheap to bring together
    (1, 512, 16, 64, 2 * 16), (3, 512, 7, 64, 3 * 16), (1, 192, 16, 64, 2 * 12), (3, 192, 7, 64, 3 * 12), (1, 48, 11, 96, 3 * 3), (2, 48, 20, 64, 12 * 3),
    # those of many are not, all 64 filters of a small launch in one workgroup apart
    (1, 512, 14, 512, 16 * 8), (1, 128, 28, 256, 28 * 4), (1, 192, 14, 512, 16 * 4), (4, 48, 14, 512, 64), (1, 48, 56, 64, 28 * 3), (1, 96, 56, 64, 28 * 3),
    (8, 384, 10, 256, 48 * 5), (3, 512, 14, 512, 48 * 5),
])
def test_packed_conv_splits_of_the_rule(device, N, C, hw, F, workgroups):
    _, _, grid, _ = _recorded(device, N, C, hw, hw, F, 3)
    assert grid[0] == workgroups
    x, w, bias = _operands(7, N, C, hw, hw, F)
    assert_close(_run(device, x, w, bias, [1, 1, 1, 1], 3, times=2), _oracle(x, w, bias, [1, 1, 1, 1]), what="three parts")


def test_packed_conv_layouts(device):
    x, w, bias = _operands(8, 2, 24, 11, 18, 40)
    want = _oracle(x, w, bias, [1, 1, 1, 1])
    rng = np.random.default_rng(9)
    for lx, lw, lo in zip(some_layouts(4, rng), some_layouts(4, rng)[::-1], some_layouts(4, rng)):
        assert_close(_run(device, x, w, bias, [1, 1, 1, 1], 3, layouts=(lx, lw, lo)), want, what=f"{lx} {lw} {lo}")


@pytest.mark.parametrize("splits", [1, 2])
def test_packed_conv_outside_the_parts(device, splits):
    """Infinities and NaN behave as in fp32, and operands whose parts would be denormal keep their precision."""
    x, w, bias = _operands(10, 1, 32, 12, 18, 64)
    x[0, 3, 4, 5], x[0, 30, 9, 0] = np.inf, np.nan
    w[2, 1, 1, 1] = -np.inf
    with np.errstate(invalid="ignore"):
        want = _oracle(x, w, bias, [1, 1, 1, 1], relu=False)
    got = _run(device, x, w, bias, [1, 1, 1, 1], 3, splits=splits, chain=[])
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    fine = np.isfinite(want)
    assert_close(got[fine], want[fine], what="finite results beside infinities")
    x, w, _ = _operands(11, 1, 32, 12, 18, 64)
    x = np.abs(x) * np.float32(1e-36)
    got = _run(device, x, np.abs(w), None, [1, 1, 1, 1], 3, splits=splits, chain=[])
    want = _oracle(x, np.abs(w), None, [1, 1, 1, 1], relu=False)
    np.testing.assert_allclose(got, want, rtol=1e-5)


def test_packed_conv_is_as_exact_as_fp32(device):
    x, w, _ = _operands(12, 1, 512, 14, 14, 64)
    pads = [1, 1, 1, 1]
    got = _run(device, x, w, None, pads, 3, chain=[]).astype(np.float64)
    padded = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (1, 1), (1, 1)))
    want = np.zeros(got.shape)
    for kh in range(3):
        for kw in range(3):
            want[0] += np.einsum("fc,chw->fhw", w[:, :, kh, kw].astype(np.float64), padded[0, :, kh:kh + 14, kw:kw + 14])
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < 3e-7  # (fp32 sums of 4608 products: 4e-7 .. 1.2e-6)


@pytest.mark.parametrize("fuse", ["1", "0"])
@pytest.mark.parametrize("bf16", [False, True])
def test_weights_that_other_operations_read_too(device, tmp_path, monkeypatch, fuse, bf16):
    """One initializer read by the convolution the packed form is for, by ones with another stride or dilation, by a
    convolution of another tensor and by an Add."""
    from fluidml_amd import fluidml, models

    monkeypatch.setenv("FLUIDML_FUSE", fuse)
    net = models.Net("shared", 3)
    w = net.normal((32, 32, 3, 3), std=0.06)
    x = net.input("x", np.float32, (1, 32, 13, 15))
    z = net.input("z", np.float32, (32, 32, 3, 3))
    y = net.input("y", np.float32, (2, 32, 9, 20))
    net.output(net.relu(net.conv(x, w, None, [1, 1], [1, 1, 1, 1])))
    net.output(net.relu(net.conv(x, w, None, [2, 2], [1, 1, 1, 1])))
    net.output(net.relu(net.conv(x, w, None, [1, 1], [2, 2, 2, 2], dilations=[2, 2])))
    net.output(net.conv(x, w, None, [2, 1], [0, 0, 0, 0]))
    net.output(net.relu(net.conv(y, w, None, [1, 1], [0, 0, 0, 0])))
    net.output(net.add(z, w))
    rng = np.random.default_rng(4)
    feeds = {v.name: rng.standard_normal(v.shape, np.float32) for v in net.inputs}
    want = graph_runner.run_graph(net, feeds)
    ex = fluidml.Executor.make_plain_greedy("shared")
    ex.context().set_bf16(bf16)
    ex.compile(net.save(os.path.join(tmp_path, "shared.onnx")))
    outs = {v.name: np.full(v.shape, 9.0, np.float32) for v in net.outputs}
    print("[case]", fuse, bf16, flush=True)
    ex.invoke({**feeds, **outs})
    for i, v in enumerate(net.outputs):
        if bf16 and i < 5:  # 288 products of operands rounded to 8 bits: 2^-9 each way, results about 1.7
            assert np.abs(outs[v.name] - want[v.name]).max() < 0.06, i
        else:
            assert_close(outs[v.name], want[v.name], what=f"output {i}")


@pytest.mark.parametrize("tile,splits", [(1, 1), (2, 1), (1, 2)])
def test_packed_conv_products_that_vanish(device, tile, splits):
    """Results of denormal numbers (see test_packed_products_that_vanish), and zeros where the input has nothing else."""
    x, w, _ = _operands(13, 1, 32, 12, 40, 64)
    for x_scale, w_scale in ((1e-42, 1.0), (1e-26, 1e-16)):
        tiny, weights = ((np.abs(x) + 0.5).astype(np.float64) * x_scale).astype(np.float32), (np.abs(w) + np.float32(0.5)) * np.float32(w_scale)
        tiny[..., 20:] = 0
        want = _oracle(tiny.astype(np.float32), weights, None, [1, 1, 1, 1], relu=False)
        got = _run(device, tiny, weights, None, [1, 1, 1, 1], 3, tile, splits, chain=[])
        assert want.max() > 0 and (np.abs(got.astype(np.float64) - want) <= 2 * 288 * 2.0 ** -150 + 1e-5 * want).all()  # (both round)
        assert (got[..., 21:] == 0).all()


def test_conv_weights_the_parts_cannot_carry(device, tmp_path):
    """Refused by the library, left as they stand by a plan."""
    from fluidml_amd import cabi, fluidml, models

    x, w, bias = _operands(14, 1, 32, 12, 18, 64)
    for value in (2.0 ** -61, 1e-40, 2.0 ** 20):
        v = w.copy()
        v[63, 31, 2, 2] = value
        with pytest.raises(cabi.FluidmlHipError) as e:
            _run(device, x, v, bias, [1, 1, 1, 1], 3)
        assert e.value.code == cabi.FL_ERR_UNSUPPORTED
        net = models.Net("refused", 3)
        net.output(net.relu(net.conv(net.input("x", np.float32, x.shape), net.const(v), net.const(bias), [1, 1], [1, 1, 1, 1])))
        ex = fluidml.Executor.make_plain_greedy("refused")
        ex.compile(net.save(os.path.join(tmp_path, "refused.onnx")))
        out = np.zeros(net.outputs[0].shape, np.float32)
        ex.invoke({"x": x, net.outputs[0].name: out})
        assert_close(out, _oracle(x, v, bias, [1, 1, 1, 1]), what=str(value))

"""3x3 convolutions that deliver the maxima of 2 x 2 windows (fluidml_hip_conv3x3_packed_chain_pool): bit for bit the pool over
the convolution's own result, and the launch a compiled graph makes of Conv, Relu and MaxPool."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def ref(t):
    from fluidml_amd import cabi

    return ctypes.byref(cabi.make_tensor(t.data_ptr(), cabi.FL_FLOAT32, t.shape, t.stride()))


@pytest.mark.parametrize("N,C,H,W,F,pads", [
    (1, 16, 8, 16, 128, [1, 1, 1, 1]),   # one workgroup
    (2, 32, 9, 17, 65, [1, 1, 1, 1]),    # one row and one column in no window, one past every tile
    (1, 48, 7, 15, 127, [1, 1, 1, 1]),
    (1, 17, 10, 20, 32, [0, 0, 0, 0]),
    (1, 5, 4, 4, 33, [0, 0, 0, 0]),      # one window
    (3, 31, 5, 33, 96, [2, 0, 1, 2]),
    (1, 160, 6, 6, 160, [1, 1, 1, 1]),   # split by the library's rule
    (5, 16, 67, 70, 130, [1, 1, 1, 1]),  # more than two workgroups to a compute unit (with two tiles per wave): another kernel without the pool
    (7, 9, 66, 129, 64, [1, 1, 1, 1]),
])
@pytest.mark.parametrize("tile,splits", [(0, 0), (1, 3), (2, 2)])
@pytest.mark.parametrize("last", [False, True], ids=["planes", "channels_last"])
def test_conv_pool(device, N, C, H, W, F, pads, tile, splits, last):
    import torch

    from fluidml_amd import cabi

    print("[case]", N, C, H, W, F, pads, tile, splits, last, flush=True)
    g = torch.Generator(device=device)
    g.manual_seed(C + F + W)
    x, w, b = (torch.randn(*s, device=device, generator=g) for s in ((N, C, H, W), (F, C, 3, 3), (F,)))
    x[-1, 0, 1, 1] = float("nan")
    OH, OW = H + pads[0] + pads[2] - 2, W + pads[1] + pads[3] - 2
    form = torch.channels_last if last else torch.contiguous_format
    for parts, chain in ((3, [(cabi.EW_RELU, 0.0)]), (1, [])):
        size = ctypes.c_size_t()
        cabi.call("conv3x3_packed_bytes", ref(w), parts, ctypes.byref(size))
        packed = torch.zeros(size.value, dtype=torch.uint8, device=device)
        cabi.call("conv3x3_pack", ref(w), parts, packed.data_ptr(), None)
        whole = torch.full((N, F, OH, OW), 9.0, device=device)
        pooled = torch.full((N, F, OH // 2, OW // 2), 9.0, device=device).contiguous(memory_format=form)
        for name, out in (("conv3x3_packed_chain", whole), ("conv3x3_packed_chain_pool", pooled)):
            for _ in range(2):  # (again: the arrival counters of a split launch are back at zero)
                cabi.call(name, ref(x), ref(w), packed.data_ptr(), parts, ref(b), ref(out), cabi.i64_array(pads),
                          ctypes.byref(cabi.make_chain(chain)), tile << 4 | splits << 8, None)
        want = torch.nn.functional.max_pool2d(whole.cpu(), 2)
        assert torch.equal(pooled.isnan().cpu(), want.isnan()) and want.isnan().any() == whole[..., :OH // 2 * 2, :OW // 2 * 2].isnan().any().cpu()
        assert torch.equal(pooled.cpu().nan_to_num(7.0), want.nan_to_num(7.0))


def test_conv_without_pool_fits(device):
    """The pooled epilogue takes bf16 launches of many workgroups without a pool none of their registers."""
    import torch

    from fluidml_amd import cabi
    from util import launches

    x, w, b, out = (torch.zeros(*s, device=device) for s in ((4, 64, 112, 112), (128, 64, 3, 3), (128,), (4, 128, 112, 112)))
    size = ctypes.c_size_t()
    cabi.call("conv3x3_packed_bytes", ref(w), 1, ctypes.byref(size))
    packed = torch.zeros(size.value, dtype=torch.uint8, device=device)
    call = lambda s: cabi.call("conv3x3_packed_chain", ref(x), ref(w), packed.data_ptr(), 1, ref(b), ref(out), cabi.i64_array([1] * 4),
                               ctypes.byref(cabi.make_chain([])), 1 << 4 | 1 << 8, s)  # (two tiles per wave: 784 workgroups)
    call(None)
    (name, fit), = launches(call)
    assert "ConvPartsKernel" in name and fit >= 3


@pytest.mark.parametrize("packed", ["1", "0"])
def test_graph_conv_pool(device, tmp_path, monkeypatch, packed):
    """The launch takes the pool with it, also where the weights are not packed (two kernels then), and gives the same."""
    from fluidml_amd import fluidml, models

    g = models.Net("conv_pool", 3)
    x = g.input("x", np.float32, (2, 16, 22, 19))
    w = [g.he_normal((48, 16, 3, 3), fan_in=144), g.he_normal((64, 48, 3, 3), fan_in=432)]
    x = g.max_pool(g.relu(g.conv(x, w[0], g.const(np.linspace(-1, 1, 48, dtype=np.float32)), [1, 1], [1, 1, 1, 1])), [2, 2], [2, 2])
    x = g.max_pool(g.relu(g.conv(x, w[1], None, [1, 1], [1, 1, 1, 1])), [2, 2], [2, 2])
    g.output(g.unary("Tanh", x))
    path = g.save(str(tmp_path / "net.onnx"))
    feed = np.random.default_rng(4).standard_normal((2, 16, 22, 19), np.float32)
    monkeypatch.setenv("FLUIDML_CONV_PACKED", packed)
    results, launches = {}, {}
    for pool in ("1", "0"):
        monkeypatch.setenv("FLUIDML_CONV_POOL", pool)
        print("[case] conv and pool, FLUIDML_CONV_PACKED =", packed, "FLUIDML_CONV_POOL =", pool, flush=True)
        ex = fluidml.Executor.make_plain_greedy("pool" + pool)
        ex.compile(path)
        for _ in range(3):
            out = {v.name: np.zeros(v.shape, np.float32) for v in g.outputs}
            ex.invoke({"x": feed, **out})
        (results[pool],) = out.values()
        launches[pool] = [t["kernel"] for t in ex.profile(1, 1)]
    assert sum("Conv" in k and "MaxPool" in k for k in launches["1"]) == 2, launches["1"]
    assert not any("Conv" in k and "MaxPool" in k for k in launches["0"]), launches["0"]
    assert np.array_equal(results["1"], results["0"])

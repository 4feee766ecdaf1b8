"""Convolutions of short sums against the float64 convolution: what conv_short.hip takes (every number of matrix steps, runs of four
pixels and single ones, image edges on both sides of a run, strides, dilations, more filters than a wave holds, several images, rows
and planes apart), what it leaves to the other kernels, and the line between them."""
import ctypes

import pytest

from test_gpu_matmul_parts import close
from util import launches

pytestmark = pytest.mark.gpu


def ref(t):
    from fluidml_amd import cabi

    return ctypes.byref(cabi.make_tensor(t.data_ptr(), cabi.FL_FLOAT32, t.shape, t.stride()))


# images, channels, filters, height, width, kernel, strides, dilations, pads
CASES = [
    (1, 3, 64, 24, 32, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),     # four in a row, both edges
    (2, 3, 64, 9, 12, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),      # the last run of pixels ragged
    (2, 3, 70, 11, 13, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),     # odd width: single pixels; filters past a wave's
    (1, 3, 32, 33, 30, (3, 3), (2, 2), (1, 1), (1, 1, 1, 1)),     # stride 2
    (1, 3, 16, 12, 20, (3, 3), (2, 1), (1, 1), (0, 1, 0, 1)),     # stride along the rows alone
    (1, 3, 33, 10, 16, (3, 3), (1, 1), (1, 1), (2, 2, 2, 2)),     # two columns past the image
    (1, 3, 16, 10, 16, (3, 3), (1, 1), (2, 3), (2, 3, 2, 3)),     # dilated
    (3, 1, 16, 8, 8, (5, 5), (1, 1), (1, 1), (0, 0, 0, 0)),       # no padding
    (1, 2, 5, 7, 6, (2, 2), (1, 1), (1, 1), (0, 0, 0, 0)),        # 8 terms, width 4 + ...
    (1, 2, 40, 4, 4, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),       # 18 terms, a row is one run
    (1, 8, 16, 6, 9, (2, 2), (1, 1), (1, 1), (1, 0, 0, 1)),       # 32 terms, uneven padding
    (1, 4, 1, 1, 40, (1, 7), (1, 1), (1, 1), (0, 3, 0, 3)),       # one row, one filter
    (1, 1, 64, 3, 3, (3, 3), (1, 1), (1, 1), (0, 0, 0, 0)),       # one pixel
]


# (few of these reach conv_short.hip: unit stride along the columns, images from width 4, at most one column of padding on the left,
# and from the second on 144 waves)
SHORT = [
    (1, 3, 64, 72, 66, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),      # four in a row and a last pair, both edges
    (4, 3, 70, 35, 31, (3, 3), (1, 1), (2, 3), (2, 1, 2, 1)),      # dilated both ways; odd width; filters past a wave's
    (4, 1, 33, 70, 50, (5, 5), (2, 1), (1, 1), (0, 0, 0, 0)),      # 25 terms, stride along the rows
    (5, 2, 5, 60, 41, (2, 2), (1, 1), (1, 1), (0, 0, 0, 0)),       # 8 terms, few filters
    (1, 8, 130, 45, 44, (2, 2), (1, 1), (1, 2), (1, 0, 0, 1)),     # 32 terms, uneven padding
    (2, 4, 1, 1, 5000, (1, 7), (1, 1), (1, 1), (0, 1, 0, 3)),      # one row, one filter
    (6, 4, 20, 75, 70, (7, 1), (3, 1), (2, 1), (3, 0, 4, 0)),      # one column of taps
    (40, 3, 32, 17, 16, (3, 1), (1, 1), (1, 1), (1, 0, 1, 0)),
    (300, 1, 64, 6, 4, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),      # a row is one run
    (1, 1, 16, 100, 100, (1, 2), (1, 1), (1, 3), (0, 1, 0, 4)),    # two terms; whole runs past the right edge
]


def apart(t):
    """The same tensor with channels outermost, rows two elements apart and planes five more."""
    import torch

    n, c, h, w = t.shape
    held = torch.full((c, n, h * (w + 2) + 5), 9.0, device=t.device)
    view = held.as_strided((n, c, h, w), (held.stride(1), held.stride(0), w + 2, 1))
    view.copy_(t)
    return view


def conv(x, w, b, out, case):
    from fluidml_amd import cabi

    strides, dilations, pads = case[6:]
    relu = cabi.make_chain([(cabi.EW_RELU, 0.0)])
    return lambda s: cabi.call("conv_chain", ref(x), ref(w), ref(b), ref(out), cabi.i64_array(pads), cabi.i64_array(strides),
                               cabi.i64_array(dilations), ctypes.c_int64(1), ctypes.byref(relu), ctypes.c_uint32(0), s)


def check(device, case, form):
    """Runs the case against float64; the kernel's name."""
    import torch

    N, C, F, H, W, kernel, strides, dilations, pads = case
    print("[case]", case, form, flush=True)
    g = torch.Generator(device=device)
    g.manual_seed(C + F + W)
    x, w, b = (torch.randn(*s, device=device, generator=g) for s in ((N, C, H, W), (F, C) + kernel, (F,)))
    x[0, 0, 0, 0] = 40.0
    want = torch.nn.functional.pad(x.double().cpu(), (pads[1], pads[3], pads[0], pads[2]))
    want = torch.nn.functional.conv2d(want, w.double().cpu(), b.double().cpu(), strides, 0, dilations).clamp_min(0)
    out = torch.full(want.shape, 9.0, device=device)
    if form == "channels_last":
        x, w, out = (t.to(memory_format=torch.channels_last) for t in (x, w, out))
    elif form == "apart":
        x, w, out = apart(x), w.to(memory_format=torch.channels_last), apart(out)
    call = conv(x, w, b, out, case)
    call(None)
    close(out, want, "conv")
    (name, _), = launches(call)
    return name


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])) + "k" + "x".join(map(str, c[5])))
@pytest.mark.parametrize("last", [False, True], ids=["planes", "channels_last"])
def test_conv_short(device, case, last):
    check(device, case, "channels_last" if last else "planes")


@pytest.mark.parametrize("case", SHORT, ids=lambda c: "x".join(map(str, c[:5])) + "k" + "x".join(map(str, c[5])))
@pytest.mark.parametrize("form", ["planes", "apart"])
def test_conv_short_reached(device, case, form):
    assert "ConvShortKernel" in check(device, case, form)


@pytest.mark.parametrize("N,F,H,W,kernel,short", [
    (1, 32, 97, 97, (2, 2), True), (1, 32, 97, 96, (2, 2), False), (1, 1, 97, 97, (2, 2), True), (1, 1, 96, 97, (2, 2), False),
    (8, 33, 24, 25, (2, 2), False), (9, 33, 24, 25, (2, 2), True), (1, 128, 48, 49, (1, 2), True), (1, 128, 47, 49, (1, 2), False),
    (1, 8, 8, 8, (3, 3), True),  # (instead of the kernel that stages a patch)
])
def test_conv_short_rule(device, N, F, H, W, kernel, short):
    """144 waves of 64 pixels and 32 filters."""
    import torch

    case = (N, 2, F, H, W, kernel, (1, 1), (1, 1), (0, 0, 0, 0))
    x, w, b = (torch.zeros(*s, device=device) for s in ((N, 2, H, W), (F, 2) + kernel, (F,)))
    out = torch.zeros(N, F, H - kernel[0] + 1, W - kernel[1] + 1, device=device)
    # (that kernel does not take weights whose channels come last)
    for weights, expected in ((w, short), (w.to(memory_format=torch.channels_last), short and kernel != (3, 3))):
        call = conv(x, weights, b, out, case)
        call(None)
        (name, _), = launches(call)
        assert ("ConvShortKernel" in name) == expected


def test_conv_short_switch(device, monkeypatch):
    """FLUIDML_CONV_HALO=0 is about kernels of 3 x 3."""
    monkeypatch.setenv("FLUIDML_CONV_HALO", "0")
    assert "ConvShortKernel" not in check(device, SHORT[0], "planes")
    assert "ConvShortKernel" in check(device, SHORT[4], "planes")


def test_conv_short_edges_hold_no_infinity(device):
    """What a run reads beside the image's edge belongs to another row or term and reaches no result."""
    import torch

    from fluidml_amd import cabi

    for W in (8, 9):
        x = torch.zeros(1, 3, 4, W, device=device)
        x[0, :, 1, :] = float("inf")  # seen by the rows 0 .. 2 of the result
        w = torch.ones(8, 3, 3, 3, device=device)
        out = torch.full((1, 8, 4, W), 9.0, device=device)
        cabi.call("conv_chain", ref(x), ref(w), None, ref(out), cabi.i64_array([1] * 4), cabi.i64_array([1, 1]), cabi.i64_array([1, 1]),
                  ctypes.c_int64(1), ctypes.byref(cabi.make_chain([])), ctypes.c_uint32(0), None)
        assert out[:, :, :3].isinf().all() and (out[:, :, 3] == 0).all()

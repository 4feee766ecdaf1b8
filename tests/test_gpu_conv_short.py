"""Convolutions of short sums (conv_short.hip) against the float64 convolution: every number of matrix steps, runs of four pixels and
single ones, image edges on both sides of a run, strides, dilations, more filters than a wave holds, several images, layouts."""
import ctypes

import pytest

from test_gpu_matmul_parts import close

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


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])) + "k" + "x".join(map(str, c[5])))
@pytest.mark.parametrize("last", [False, True], ids=["planes", "channels_last"])
def test_conv_short(device, case, last):
    import torch

    from fluidml_amd import cabi

    N, C, F, H, W, kernel, strides, dilations, pads = case
    print("[case]", case, last, flush=True)
    g = torch.Generator(device=device)
    g.manual_seed(C + F + W)
    x, w, b = (torch.randn(*s, device=device, generator=g) for s in ((N, C, H, W), (F, C) + kernel, (F,)))
    x[0, 0, 0, 0] = 40.0
    want = torch.nn.functional.pad(x.double().cpu(), (pads[1], pads[3], pads[0], pads[2]))
    want = torch.nn.functional.conv2d(want, w.double().cpu(), b.double().cpu(), strides, 0, dilations).clamp_min(0)
    if last:
        x, w = (t.to(memory_format=torch.channels_last) for t in (x, w))
    out = torch.full(want.shape, 9.0, device=device).contiguous(memory_format=torch.channels_last if last else torch.contiguous_format)
    relu = cabi.make_chain([(cabi.EW_RELU, 0.0)])
    cabi.call("conv_chain", ref(x), ref(w), ref(b), ref(out), cabi.i64_array(pads), cabi.i64_array(strides), cabi.i64_array(dilations),
              ctypes.c_int64(1), ctypes.byref(relu), ctypes.c_uint32(0), None)
    close(out, want, "conv")


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

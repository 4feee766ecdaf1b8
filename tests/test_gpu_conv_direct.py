"""Depthwise convolutions whose taps are requested together (one thread per output, windows known at compile time): taps beside the
input, on both sides at once too, take no part, not even those next to an infinity."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


def ref(t):
    from fluidml_amd import cabi

    return ctypes.byref(cabi.make_tensor(t.data_ptr(), cabi.FL_FLOAT32, t.shape, t.stride()))


# images, channels, extents, window, strides, dilations, pads (before, after)
CASES = [
    (1, 768, (128,), (9,), (1,), (1,), (4, 4)),
    (2, 5, (4,), (9,), (1,), (1,), (4, 4)),       # every output misses taps on both sides
    (3, 7, (33,), (9,), (2,), (3,), (0, 13)),
    (2, 9, (17,), (3,), (1,), (5,), (5, 5)),
    (2, 2, (3,), (3,), (1,), (1,), (0, 0)),       # one output a channel
    (2, 3, (60, 51), (3, 3), (2, 1), (1, 2), (1, 2, 0, 3)),
    (1, 4, (50, 3), (5, 5), (1, 2), (1, 1), (2, 2, 2, 2)),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[2])) + "k" + "x".join(map(str, c[3])))
@pytest.mark.parametrize("last", [False, True], ids=["planes", "channels_last"])
def test_conv_direct(device, monkeypatch, case, last):
    import torch

    from fluidml_amd import cabi

    monkeypatch.setenv("FLUIDML_CONV_PLANE", "0")
    N, C, extents, window, strides, dilations, pads = case
    print("[case]", case, last, flush=True)
    g = torch.Generator(device=device)
    g.manual_seed(C)
    x, w, b = (torch.randn(*s, device=device, generator=g) for s in ((N, C) + extents, (C, 1) + window, (C,)))
    x[0, 0].view(-1)[0] = float("inf")
    ns = len(extents)
    widths = [v for d in reversed(range(ns)) for v in (pads[d], pads[d + ns])]
    conv = torch.nn.functional.conv1d if ns == 1 else torch.nn.functional.conv2d
    # (zero beside the input: an infinity there would be a tap that takes part)
    want = conv(torch.nn.functional.pad(x.double().cpu(), widths), w.double().cpu(), b.double().cpu(), strides, 0, dilations, C)
    out = torch.full(want.shape, 9.0, device=device)
    if last:
        x, out = (t.movedim(1, -1).contiguous().movedim(-1, 1) for t in (x, out))
    cabi.call("conv_chain", ref(x), ref(w), ref(b), ref(out), cabi.i64_array(pads), cabi.i64_array(strides), cabi.i64_array(dilations),
              ctypes.c_int64(C), ctypes.byref(cabi.make_chain([])), ctypes.c_uint32(0), None)
    got = out.double().cpu()
    fine = want.isfinite()
    assert torch.equal(got.isfinite(), fine) and torch.equal(got[~fine].sign(), want[~fine].sign())
    # a sum of n terms up to |x| |w| <= 25 with one rounding each, and the bias
    n = 1
    for k in window:
        n *= k
    assert (got - want)[fine].abs().max() <= 2.0 ** -24 * 25 * n * (n + 1)

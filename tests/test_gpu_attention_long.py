"""Fused attention with more than 256 keys on the GPU, at the edges of its key chunks and row groups, against the
oracle's chain of MatMul, Div, Add, Where, Softmax and MatMul."""
import ctypes

import numpy as np
import pytest

from oracle import kernels as ok
from tests.util import DeviceView, assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,sq,skv,d,masked,where", [
    (12, 512, 512, 64, True, False),   # two row groups per workgroup, 128-bit loads
    (8, 500, 388, 64, True, True),     # three chunks, the last nearly empty
    (16, 257, 257, 32, False, True),   # one key past two chunks, one row past a workgroup, scalar loads
    (2, 40, 384, 64, True, False),     # too few workgroups for two groups
    (1, 17, 511, 61, True, True),
    (64, 33, 385, 8, False, False),
])
def test_attention_long(device, heads, sq, skv, d, masked, where):
    from fluidml_amd import cabi

    rng = np.random.default_rng(sq + skv)
    draw = lambda *shape: rng.uniform(-1, 1, shape).astype(np.float32)  # noqa: E731
    q, kt, v = draw(heads, sq, d), draw(heads, d, skv), draw(heads, skv, d)
    mask = rng.uniform(-8, 0, (1, 1, skv)).astype(np.float32) if masked else None
    cond = np.tril(np.ones((sq, skv), np.bool_), skv - sq)[None] if where else None
    fill = float(np.finfo(np.float32).min)
    s = ok.View.empty((heads, sq, skv))
    ok.matmul(ok.View(q), ok.View(kt), s)
    t = ok.View.empty(s.shape)
    ok.unary_f32(ok.OP_DIV_C, s, t, float(np.sqrt(d)))
    if masked:
        s, t = t, ok.View.empty(s.shape)
        ok.binary_f32(ok.BOP_ADD, s, ok.View(mask), t)
    if where:
        s, t = t, ok.View.empty(s.shape)
        ok.where(ok.View(cond), s, None, fill, t)
    p, want = ok.View.empty(s.shape), ok.View.empty((heads, sq, d))
    ok.softmax(t, p, 2)
    ok.matmul(p, ok.View(v), want)
    print("[case]", heads, sq, skv, d, flush=True)
    dq, dk, dv, do = (DeviceView(x, device) for x in (ok.View(q), ok.View(kt), ok.View(v), ok.View.empty(want.shape, fill=3)))
    dm, dc = DeviceView(ok.View(mask), device) if masked else None, DeviceView(ok.View(cond), device) if where else None
    cabi.call("attention", dq.ref(), dk.ref(), dv.ref(), do.ref(), ctypes.c_double(np.sqrt(d)), 1, dm.ref() if dm else None,
              dc.ref() if dc else None, ctypes.c_double(fill), None)
    assert_close(do.logical(), want.logical(), what="attention")

"""Fused attention with more than 256 keys on the GPU (eight waves share a query block's keys, 64 each; a block is 16
queries), at the edges of waves and blocks, against the oracle's chain of MatMul, Div, Add, Where, Softmax and MatMul."""
import ctypes

import numpy as np
import pytest

from oracle import kernels as ok
from tests.util import DeviceView, assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,sq,skv,d,masked,where", [
    (12, 512, 512, 64, True, False),   # all waves full
    (8, 500, 388, 64, True, True),     # the seventh wave has four keys, the eighth none; four queries in the last block
    (16, 257, 257, 32, False, True),   # one key in the fifth wave, none in three; one query in the last block
    (2, 40, 384, 64, True, False),     # six full waves, two without a key
    (1, 17, 511, 61, True, True),      # one key short; head columns that no wide load fits
    (64, 33, 385, 8, False, False),    # half a tile of head columns; one key in the seventh wave
])
def test_attention_long(device, heads, sq, skv, d, masked, where):
    rng = np.random.default_rng(sq + skv)
    draw = lambda *shape: rng.uniform(-1, 1, shape).astype(np.float32)  # noqa: E731
    q, kt, v = draw(heads, sq, d), draw(heads, d, skv), draw(heads, skv, d)
    mask = rng.uniform(-8, 0, (1, 1, skv)).astype(np.float32) if masked else None
    cond = np.tril(np.ones((sq, skv), np.bool_), skv - sq)[None] if where else None
    print("[case]", heads, sq, skv, d, flush=True)
    got, want = _both(device, q, kt, v, mask, cond, float(np.finfo(np.float32).min))
    assert_close(got, want, what="attention")


def _both(device, q, kt, v, mask, cond, fill):
    """(kernel, oracle) for q [heads, sq, d], kt [heads, d, skv], v [heads, skv, d]"""
    from fluidml_amd import cabi

    heads, sq, d = q.shape
    skv = v.shape[1]
    s = ok.View.empty((heads, sq, skv))
    ok.matmul(ok.View(q), ok.View(kt), s)
    t = ok.View.empty(s.shape)
    ok.unary_f32(ok.OP_DIV_C, s, t, float(np.sqrt(d)))
    if mask is not None:
        s, t = t, ok.View.empty(s.shape)
        ok.binary_f32(ok.BOP_ADD, s, ok.View(mask), t)
    if cond is not None:
        s, t = t, ok.View.empty(s.shape)
        ok.where(ok.View(cond), s, None, fill, t)
    p, want = ok.View.empty(s.shape), ok.View.empty((heads, sq, d))
    ok.softmax(t, p, 2)
    ok.matmul(p, ok.View(v), want)
    dq, dk, dv, do = (DeviceView(x, device) for x in (ok.View(q), ok.View(kt), ok.View(v), ok.View.empty(want.shape, fill=3)))
    dm, dc = DeviceView(ok.View(mask), device) if mask is not None else None, DeviceView(ok.View(cond), device) if cond is not None else None
    cabi.call("attention", dq.ref(), dk.ref(), dv.ref(), do.ref(), ctypes.c_double(np.sqrt(d)), 1, dm.ref() if dm else None,
              dc.ref() if dc else None, ctypes.c_double(fill), None)
    return do.logical(), want.logical()


@pytest.mark.parametrize("skv,keys", [(512, 64), (257, 64), (200, 32), (37, 16)])  # keys of a wave
@pytest.mark.parametrize("case", ["wave masked", "one wave left", "all masked", "wave filled", "all filled", "scores", "values"])
def test_attention_merges_what_is_not_finite(device, skv, keys, case):
    """Waves whose keys are all masked, by -inf or by the type's lowest value; scores that are NaN or infinite; and an
    infinity in the last key's row of V, which the lanes behind the last key read too."""
    heads, sq, d = 2, 20, 64
    rng = np.random.default_rng(skv)
    draw = lambda *shape: rng.uniform(-1, 1, shape).astype(np.float32)  # noqa: E731
    q, kt, v = draw(heads, sq, d), draw(heads, d, skv), draw(heads, skv, d)
    mask, cond, fill = np.zeros((1, 1, skv), np.float32), None, float(np.finfo(np.float32).min)
    if case == "wave masked":
        mask[..., keys:2 * keys] = -np.inf
    elif case == "one wave left":
        mask[..., :keys] = mask[..., 2 * keys:] = -np.inf
    elif case == "all masked":
        mask[:] = -np.inf
    elif case == "wave filled":
        cond = np.ones((1, sq, skv), np.bool_)
        cond[:, ::2, :keys] = cond[:, 1::2, keys:] = False
    elif case == "all filled":
        cond = np.zeros((1, sq, skv), np.bool_)
    elif case == "scores":
        q[0, 3, 5], kt[1, 7, skv - 1] = np.nan, np.inf  # (the second: plus or minus infinity, query by query)
    else:
        v[0, skv - 1, 9], v[1, 0, 60] = np.inf, -np.inf
        mask[..., 0] = -np.inf  # (nothing times an infinity)
    print("[case]", skv, case, flush=True)
    with np.errstate(invalid="ignore"):
        got, want = _both(device, q, kt, v, mask, cond, fill)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    fine = np.isfinite(want)
    assert_close(got[fine], want[fine], what=case)
